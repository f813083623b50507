"""Settings with more species than one pinned line of sizes holds: 64 to the
largest count (255), builds in one workgroup and in several. Against the
oracle; 256 species are refused."""
import numpy as np
import pytest

from helpers import random_cell, rel_err

pytestmark = pytest.mark.gpu


def check(oracle, nos, n, N, L, predict):
    from flare_amd import _C_flare as C
    rc = 3.2
    cell, species, pos = random_cell(n, nos, nos=nos, scale=2.6 * n ** (1 / 3), skew=0.1)
    cut = np.full((nos, nos), rc)
    cut[:, ::3] = 2.9
    calc = C.B2("chebyshev", "quadratic", [0.0, rc], [], [nos, N, L], cut)
    s = C.Structure(cell, species, pos, rc, [calc])
    d = s.descriptors[0]
    near = oracle.Neighbors(cell, species, pos, rc, "cells")
    centre = np.repeat(species, near.neighbor_count)
    keep = near.relative_positions[:, 0] <= cut[centre, species[near.structure_indices]]
    assert d.n_clusters_by_type == [int((species == t).sum()) for t in range(nos)]
    assert d.n_neighbors_by_type == [int(keep[centre == t].sum()) for t in range(nos)]
    assert np.array_equal(np.concatenate(d.atom_indices), np.argsort(species, kind="stable"))
    if not predict:
        return
    ref = oracle.B2Values(near, nos, N, L, cut)
    for t in set(species.tolist()):
        assert rel_err(d.descriptors[t], ref.descriptors[t]) < 1e-10
    sgp = C.SparseGP([C.NormalizedDotProduct(1.5, 2.0)], 0.01, 0.05, 0.005)
    sgp.add_specific_environments(s, list(range(0, n, 5)))
    sgp.update_L_inverse()
    sgp.set_alpha(np.random.default_rng(5).uniform(0.1, 1.0, size=sgp.n_sparse))
    cd = sgp.sparse_descriptors[0]
    model = oracle.Model(1.5, 2.0, cd.descriptors, cd.descriptor_norms, sgp.alpha, L_inv=sgp.L_inv)
    mean, _ = model.predict(ref, "mean")
    sgp.predict_mean(s)
    assert rel_err(s.mean_efs, mean) < 1e-10


@pytest.mark.parametrize("nos,N,L", [(63, 2, 0), (64, 2, 0), (100, 1, 1), (130, 1, 0)])
def test_predictions(oracle, nos, N, L):
    check(oracle, nos, 150, N, L, True)


@pytest.mark.parametrize("n", [300, 8193])
def test_largest_count(oracle, n):
    check(oracle, 255, n, 1, 0, False)


def test_refused(oracle):
    with pytest.raises(ValueError):
        check(oracle, 256, 20, 1, 0, False)
