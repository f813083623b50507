"""Force gather and per-structure sums at the edges of their groups: 16 atoms
per workgroup, 256 per chunk, structures with one atom, without bonds and
with several chunks, alone and in a batch."""
import numpy as np
import pytest

from helpers import random_cell, rel_err

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 15, 16, 17, 255, 256, 257, 600]


def structure(n):
    if n == 2:  # no bonds
        return np.eye(3) * 30.0, np.array([0, 1], np.int32), np.array([[1.0, 1, 1], [15, 15, 15]])
    return random_cell(n, 60 + n, nos=2, scale=4.4 if n == 1 else 2.3 * n ** (1 / 3), skew=0.2)


@pytest.fixture(scope="module")
def model():
    from flare_amd import _C_flare as C
    cut = np.full((2, 2), 4.2)
    calc = C.B2("chebyshev", "quadratic", [0.0, 4.2], [], [2, 4, 2], cut)
    train = C.Structure(*random_cell(40, 7, nos=2, scale=8.0, skew=0.3), 4.2, [calc])
    sgp = C.SparseGP([C.NormalizedDotProduct(2.0, 2.0)], 0.01, 0.05, 0.005)
    sgp.add_specific_environments(train, list(range(0, 40, 3)))
    sgp.update_L_inverse()
    sgp.set_alpha(np.random.default_rng(2).normal(scale=0.1, size=sgp.n_sparse))
    return C, calc, cut, sgp


def test_forces_and_sums(oracle, model):
    from flare_amd.batch import Batch
    C, calc, cut, sgp = model
    structs = [structure(n) for n in SIZES]
    means, _ = Batch(structs, 4.2, calc).predict(sgp)
    cd = sgp.sparse_descriptors[0]
    ref = oracle.Model(2.0, 2.0, cd.descriptors, cd.descriptor_norms, sgp.alpha, L_inv=sgp.L_inv)
    for n, st, mean in zip(SIZES, structs, means):
        want, _ = ref.predict(oracle.B2Values(oracle.Neighbors(*st, 4.2), 2, 4, 2, cut), "mean")
        assert rel_err(mean, want) < 1e-10, n
        alone = C.Structure(*st, 4.2, [calc])
        sgp.predict_mean(alone)
        assert np.array_equal(alone.mean_efs, mean), n


def test_sums_of_large_and_small(model):
    """Structures of up to 2,048 atoms are summed in one launch, a batch with a
    larger one in two: the same bits either way."""
    from flare_amd.batch import Batch
    C, calc, cut, sgp = model
    structs = [structure(n) for n in (2048, 2049, 1025, 3)]
    means, _ = Batch(structs, 4.2, calc).predict(sgp)
    for st, mean in zip(structs, means):
        alone = C.Structure(*st, 4.2, [calc])
        sgp.predict_mean(alone)
        assert np.array_equal(alone.mean_efs, mean)


def test_batch_of_very_many(model):
    """12,000 structures, whose cells and offsets exceed the staging buffer."""
    from flare_amd.batch import Batch
    C, calc, cut, sgp = model
    structs = [structure(n) for n in (1, 2, 15, 3)]
    few, _ = Batch(structs, 4.2, calc).predict(sgp)
    many, _ = Batch(structs * 3000, 4.2, calc).predict(sgp)
    for k, mean in enumerate(many):
        assert np.array_equal(mean, few[k % 4]), k
