"""The chosen form's contractions at both of their tile sizes: few tiles and
many, an odd and an even number of 64-column tiles, column counts at and past a tile's
edge, one to six steps of the reduction, a last row tile with one row, several
species in one launch. The chosen form against the FP64 form."""
import numpy as np
import pytest

from helpers import fcc

pytestmark = pytest.mark.gpu

SIGMA = 1.5


# (species, radial functions, l_max): d = 20, 108, 144, 312, 360 (1, 2, 3, 5
# and 6 steps of 64); cells of 4 atoms; sparse environments per species.
@pytest.mark.parametrize("settings,reps,n_sparse", [
    ((1, 4, 1), (4, 4, 4), (1,)),
    ((1, 8, 2), (13, 13, 12), (260,)),   # 8112 atoms: 64 row tiles x 5 columns of 64
    ((1, 8, 3), (13, 13, 13), (320,)),   # 8788 atoms
    ((2, 6, 3), (4, 11, 1), (64, 65)),   # 176 atoms
    ((2, 4, 9), (16, 16, 16), (129, 190)),
    # d = 1088: 576 tiles of 128 x 128 of the gradient contraction or 160 of
    # 256 x 256, one and three steps of 32.
    ((1, 16, 7), (13, 13, 12), (30,)),
    ((1, 16, 7), (13, 13, 12), (70,)),
])
def test_integer_contraction(settings, reps, n_sparse):
    from flare_amd import _C_flare as C
    nos, N, L = settings
    cut = np.full((nos, nos), 4.2)
    calc = C.B2("chebyshev", "quadratic", [0.0, 4.2], [], list(settings), cut)
    cell, species, pos = fcc(4.0, reps, 0.1, 11, nos=nos)
    train = C.Structure(cell, species, pos, 4.2, [calc])
    d = train.descriptors[0]
    atoms = [int(a) for t, m in enumerate(n_sparse) for a in d.atom_indices[t][:m]]
    if len(atoms) < sum(n_sparse):
        pytest.fail("too few atoms of a species")
    sgp = C.SparseGP([C.NormalizedDotProduct(SIGMA, 2.0)], 0.01, 0.05, 0.005)
    sgp.Kuu_jitter = 1e-4
    sgp.add_specific_environments(train, atoms)
    sgp.update_L_inverse()
    sgp.set_alpha(np.random.default_rng(5).uniform(0.1, 1.0, size=sgp.n_sparse))
    out = []
    for form in (C.FORM_FP64, C.FORM_CHOSEN):
        s = C.Structure(cell, species, pos, 4.2, [calc], form=form)
        sgp.predict_local_uncertainties(s)
        out.append((s.mean_efs, s.local_uncertainties[0]))
    (m64, v64), (m, v) = out
    # S carries 2^-34 of the largest products per k; |L_inv| <= 1e2 amplifies
    # it in Q. Forces: FP32 adjoint with split-BF16 products.
    assert abs(m[0] - m64[0]) < 1e-7 * abs(m64[0])
    assert np.max(np.abs(m[1:-6] - m64[1:-6])) < 1e-3 * np.max(np.abs(m64[1:-6]))
    assert np.max(np.abs(v - v64)) < 1e-5 * SIGMA ** 2


# 8112 and 8788 atoms: the library takes the 128-column tiles of the integer
# contraction (144 functions, 320 environments) or the 256-wide ones of the
# gradient contraction (1088 functions); 176 atoms: the smaller ones of both.
@pytest.mark.parametrize("settings,reps,n_sparse", [
    ((1, 8, 3), (13, 13, 13), (320,)),
    ((1, 16, 7), (13, 13, 12), (70,)),
    ((2, 6, 3), (4, 11, 1), (64, 65)),
])
def test_tile_sizes_bitwise(settings, reps, n_sparse, monkeypatch):
    """Both tile sizes of either contraction give the results of the one that
    the library picks, bit for bit."""
    from flare_amd import _C_flare as C
    nos = settings[0]
    calc = C.B2("chebyshev", "quadratic", [0.0, 4.2], [], list(settings), np.full((nos, nos), 4.2))
    system = fcc(4.0, reps, 0.1, 11, nos=nos)
    train = C.Structure(*system, 4.2, [calc])
    d = train.descriptors[0]
    sgp = C.SparseGP([C.NormalizedDotProduct(SIGMA, 2.0)], 0.01, 0.05, 0.005)
    sgp.Kuu_jitter = 1e-4
    sgp.add_specific_environments(train, [int(a) for t, m in enumerate(n_sparse)
                                          for a in d.atom_indices[t][:m]])
    sgp.update_L_inverse()
    sgp.set_alpha(np.random.default_rng(5).uniform(0.1, 1.0, size=sgp.n_sparse))
    out = []
    for shape in (None, "0", "1"):
        if shape:
            monkeypatch.setenv("FLARE_MI_TILE_SHAPE", shape)
        s = C.Structure(*system, 4.2, [calc], form=C.FORM_CHOSEN)
        sgp.predict_local_uncertainties(s)
        out.append((s.mean_efs, s.local_uncertainties[0]))
    for mean, var in out[1:]:
        assert np.array_equal(mean, out[0][0]) and np.array_equal(var, out[0][1])
