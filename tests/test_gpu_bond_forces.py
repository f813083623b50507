"""Bond forces at the edges of the radial groups (4 functions each, 1 to 16),
with fewer and more harmonics than lanes and more bonds than lanes."""
import numpy as np
import pytest

from helpers import random_cell, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_max,l_max", [(1, 0), (3, 1), (4, 2), (5, 6), (8, 3), (9, 7), (13, 1),
                                         (16, 4)])
def test_radial_groups(oracle, n_max, l_max):
    from flare_amd import _C_flare as C
    cut = np.array([[4.2, 3.9], [3.9, 4.0]])
    calc = C.B2("chebyshev", "quadratic", [0.0, 4.2], [], [2, n_max, l_max], cut)
    # About 75 bonds per atom, and a few.
    dense = random_cell(30, 11, nos=2, scale=5.0, skew=0.2)
    thin = random_cell(7, 12, nos=2, scale=7.0, skew=0.3)
    train = C.Structure(*dense, 4.2, [calc])
    sgp = C.SparseGP([C.NormalizedDotProduct(2.0, 2.0)], 0.01, 0.05, 0.005)
    sgp.add_specific_environments(train, list(range(0, 30, 4)))
    sgp.update_L_inverse()
    sgp.set_alpha(np.random.default_rng(3).normal(scale=0.1, size=sgp.n_sparse))
    cd = sgp.sparse_descriptors[0]
    ref = oracle.Model(2.0, 2.0, cd.descriptors, cd.descriptor_norms, sgp.alpha, L_inv=sgp.L_inv)
    for st in (dense, thin):
        want, _ = ref.predict(oracle.B2Values(oracle.Neighbors(*st, 4.2), 2, n_max, l_max, cut),
                              "mean")
        s = C.Structure(*st, 4.2, [calc])
        sgp.predict_mean(s)
        assert rel_err(s.mean_efs, want) < 1e-10
        # FP32 adjoint and two BF16 pieces of w and of the sparse set (2^-16
        # per product).
        s = C.Structure(*st, 4.2, [calc], form=C.FORM_CHOSEN)
        sgp.predict_mean(s)
        scale = max(np.max(np.abs(want[1:])), 1e-3 * abs(want[0]))
        assert np.max(np.abs(s.mean_efs[1:] - want[1:])) < 1e-3 * scale
