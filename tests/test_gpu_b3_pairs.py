"""B3 rows and forces on both sides of the pair kernels' split over waves (up
to 64 radial pairs in FP64): 1, 55, 66 and 78 pairs, fewer l-sets than waves,
atoms without bonds. Against the oracle."""
import numpy as np
import pytest

from helpers import random_cell, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("settings,n,scale", [
    ((1, 1, 0), 9, 6.0), ((1, 1, 2), 3, 30.0), ((2, 5, 1), 21, 7.0), ((1, 11, 2), 12, 6.0),
    ((3, 4, 1), 15, 6.5)])
def test_b3_pairs(oracle, settings, n, scale):
    from flare_amd import _C_flare as C
    nos = settings[0]
    cut = np.full((nos, nos), 4.2)
    calc = C.B3("chebyshev", "quadratic", [0.0, 4.2], [], list(settings), cut)
    cell, species, pos = random_cell(n, 50 + n, nos=nos, scale=scale, skew=0.2)
    s = C.Structure(cell, species, pos, 4.2, [calc])
    ref = oracle.B3Values(oracle.Neighbors(cell, species, pos, 4.2), *settings, cut)
    d = s.descriptors[0]
    for t in range(nos):
        assert rel_err(d.descriptors[t], ref.descriptors[t]) < 1e-10
        assert rel_err(d.descriptor_norms[t], ref.descriptor_norms[t]) < 1e-10
    sgp = C.SparseGP([C.NormalizedDotProduct(1.5, 2.0)], 0.01, 0.05, 0.005)
    sgp.add_specific_environments(s, list(range(min(n, 6))))
    sgp.update_L_inverse()
    sgp.set_alpha(np.random.default_rng(3).uniform(0.1, 1.0, size=sgp.n_sparse))
    cd = sgp.sparse_descriptors[0]
    m = oracle.Model(1.5, 2.0, cd.descriptors, cd.descriptor_norms, sgp.alpha, L_inv=sgp.L_inv)
    mean, _ = m.predict(ref, "mean")
    sgp.predict_mean(s)
    assert rel_err(s.mean_efs, mean) < 1e-9
