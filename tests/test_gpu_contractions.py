"""The contractions at the sizes where their tiles can go wrong: reduction
lengths below one MFMA step, odd ones and ones just past a step; row and
column counts of 1, at a tile's edge and past it; species without atoms or
sparse environments. Against the oracle, and every tile shape against the one
the library picks, bit for bit."""
import numpy as np
import pytest

from helpers import random_cell, rel_err

pytestmark = pytest.mark.gpu

SIGMA = 1.5
# (descriptor settings, sparse environments per species): d = 6, 42, 60, 75,
# 275 and 544.
CASES = [
    ((3, 1, 0), (1, 16, 17)),
    ((3, 2, 1), (5, 0, 15)),
    ((1, 5, 3), (33,)),
    ((1, 5, 4), (48,)),
    ((2, 5, 4), (31, 7)),
    ((2, 8, 3), (25, 24)),
]


def setup(settings, n_sparse, power=2.0):
    from flare_amd import _C_flare as C
    nos, N, L = settings
    cut = np.full((nos, nos), 4.5)
    calc = C.B2("chebyshev", "quadratic", [0.0, 4.5], [], list(settings), cut)
    train = C.Structure(*random_cell(110, 31, nos=nos, scale=10.5, skew=0.4), 4.5, [calc])
    d = train.descriptors[0]
    atoms = [int(a) for s, m in enumerate(n_sparse) for a in d.atom_indices[s][:m]]
    sgp = C.SparseGP([C.NormalizedDotProduct(SIGMA, power)], 0.01, 0.05, 0.005)
    sgp.add_specific_environments(train, atoms)
    assert sgp.sparse_descriptors[0].n_clusters_by_type == list(n_sparse)
    sgp.update_L_inverse()
    sgp.set_alpha(np.random.default_rng(5).normal(scale=0.1, size=sgp.n_sparse))
    return C, calc, cut, sgp


def predict(C, calc, sgp, system, form=0):
    s = C.Structure(*system, 4.5, [calc], form=form)
    sgp.predict_local_uncertainties(s)
    return s.mean_efs, s.local_uncertainties[0]


@pytest.mark.parametrize("n", [1, 16, 49, 130])
@pytest.mark.parametrize("settings,n_sparse", CASES)
def test_fp64_contractions(oracle, settings, n_sparse, n, monkeypatch):
    nos = settings[0]
    C, calc, cut, sgp = setup(settings, n_sparse)
    system = random_cell(n, 40 + n, nos=nos, scale=5.0 if n == 1 else 2.2 * n ** (1 / 3), skew=0.2)
    mean, var = predict(C, calc, sgp, system)
    cd = sgp.sparse_descriptors[0]
    model = oracle.Model(SIGMA, 2.0, cd.descriptors, cd.descriptor_norms, sgp.alpha, L_inv=sgp.L_inv)
    ref, ref_var = model.predict(
        oracle.B2Values(oracle.Neighbors(*system, 4.5), *settings, cut), "local")
    assert rel_err(mean, ref) < 1e-10
    # |L_inv| <= 1 / sqrt(jitter) = 1e4 amplifies the rounding of k (d + 3
    # operations on values of at most sigma^2) in Q, and Q.Q doubles it.
    eps, d = np.finfo(float).eps, cd.n_descriptors
    tol = 2e4 * SIGMA ** 3 * np.sqrt(sgp.n_sparse) * (d + 3) * eps
    assert np.max(np.abs(var - ref_var)) < tol
    for shape in range(4):
        monkeypatch.setenv("FLARE_MI_TILE_SHAPE", str(shape))
        m2, v2 = predict(C, calc, sgp, system)
        assert np.array_equal(m2, mean) and np.array_equal(v2, var)
