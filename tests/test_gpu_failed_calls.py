"""What a refused or failed call leaves behind."""
import ctypes

import numpy as np
import pytest

from helpers import random_cell

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("settings", [(2, 4, 11), (2, 17, 3)])
def test_failed_recompute(settings):
    """Descriptors recomputed with settings that the kernels refuse: the
    structure has none then, instead of the new sizes with the earlier lists,
    and takes valid settings again."""
    from flare_amd import _C_flare as C
    from flare_amd import _lib
    L = _lib.load()
    cell, species, pos = random_cell(20, 5, nos=1, scale=6.5, skew=0.2)
    calc = C.B2("chebyshev", "quadratic", [0.0, 4.0], [], [1, 4, 3])
    s = C.Structure(cell, species, pos, 4.0, [calc])
    sgp = C.SparseGP([C.NormalizedDotProduct(1.5, 2.0)], 0.1, 0.1, 0.1)
    sgp.add_specific_environments(s, [0, 3, 7])
    sgp.update_L_inverse()
    sgp.set_alpha(np.ones(sgp.n_sparse))
    sgp.predict_local_uncertainties(s)
    before = s.mean_efs.copy()
    bad, keep = C.B2("chebyshev", "quadratic", [0.0, 4.0], [], list(settings))._settings()
    assert L.fm_structure_compute_b2(s._h, ctypes.byref(bad), 0) == _lib.FM_ERR_INVALID
    nd, per = ctypes.c_int(), np.zeros((2, 2), np.int32)
    assert L.fm_structure_b2_sizes(s._h, ctypes.byref(nd), _lib.ptr(per[0]),
                                   _lib.ptr(per[1])) == _lib.FM_ERR_STATE
    mean = np.zeros(1 + 3 * 20 + 6)
    model = sgp._model(0, s._ctx)
    assert L.fm_predict(model.h, s._h, _lib.PREDICT_MEAN, 0, _lib.ptr(mean), None,
                        None) == _lib.FM_ERR_STATE
    good, keep = calc._settings()
    _lib.check(L.fm_structure_compute_b2(s._h, ctypes.byref(good), 0))
    _lib.check(L.fm_predict(model.h, s._h, _lib.PREDICT_MEAN, 0, _lib.ptr(mean), None, None))
    assert np.array_equal(mean, before)


def test_failed_creation():
    """Structures and models that are refused while their uploads are queued do
    not disturb the ones made next from the same buffers."""
    from flare_amd import _C_flare as C
    calc = C.B2("chebyshev", "quadratic", [0.0, 4.0], [], [2, 4, 3])
    cell, species, pos = random_cell(300, 5, nos=2, scale=16.0, skew=0.2)
    want = C.Structure(cell, species, pos, 4.0, [calc])
    sgp = C.SparseGP([C.NormalizedDotProduct(1.5, 2.0)], 0.1, 0.1, 0.1)
    sgp.add_specific_environments(want, [int(a) for t in range(2)
                                         for a in np.flatnonzero(species == t)[:2]])
    sgp.update_L_inverse()
    sgp.set_alpha(np.linspace(-0.2, 0.3, sgp.n_sparse))
    sgp.predict_local_uncertainties(want)
    L_inv = sgp.L_inv.copy()
    for _ in range(20):
        bad = pos.copy()
        bad[17, 1] = np.nan
        with pytest.raises(ValueError):
            C.Structure(cell * 1.1, species, bad, 4.0, [calc])
        with pytest.raises(ValueError):
            C.Structure(cell * 1.1, -species - 1, pos, 4.0, [calc])
        s = C.Structure(cell, species, pos, 4.0, [calc])
        wrong = L_inv.copy()
        wrong[0, -1] = 1.0  # above the diagonal block of the second species
        sgp.L_inv = wrong
        sgp._invalidate()
        with pytest.raises(ValueError):
            sgp.predict_local_uncertainties(s)
        sgp.L_inv = L_inv
        sgp._invalidate()
        sgp.predict_local_uncertainties(s)
        assert np.array_equal(s.mean_efs, want.mean_efs)
        assert np.array_equal(s.local_uncertainties[0], want.local_uncertainties[0])
