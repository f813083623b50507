"""Derivatives and kernel matrices of the training path where their kernels
can go wrong: one and four waves per block, atoms without bonds and with more
than a wave's lanes, species without atoms or sparse environments, one, 64 and
65 environments. Against the oracle."""
import numpy as np
import pytest

from helpers import random_cell, rel_err

pytestmark = pytest.mark.gpu


# (species, radial functions, l_max), atoms, cutoff, sparse environments
@pytest.mark.parametrize("settings,n,rc,n_sparse", [
    ((1, 4, 2), 1, 3.0, (1,)),             # no bonds
    ((1, 4, 2), 1, 5.0, (1,)),             # bonds to its own images
    ((1, 3, 0), 65, 4.0, (65,)),
    ((2, 4, 3), 130, 4.0, (64, 0)),
    ((3, 2, 1), 5, 6.5, (1, 0, 2)),
    ((4, 16, 6), 9, 4.0, (2, 1, 2, 1)),    # one wave per block
])
@pytest.mark.parametrize("power", [1.0, 2.0, 3.0])
def test_training_edges(oracle, settings, n, rc, n_sparse, power):
    from flare_amd import _C_flare as C
    nos = settings[0]
    cut = np.full((nos, nos), rc)
    calc = C.B2("chebyshev", "quadratic", [0.0, rc], [], list(settings), cut)
    cell, species, pos = random_cell(n, 70 + n, nos=nos, scale=3.4 if n == 1 else 2.3 * n ** (1 / 3),
                                     skew=0.2)
    if n == 9:
        species = np.array([0, 0, 0, 1, 1, 2, 2, 3, 3], np.int32)
    if n == 5:
        species = np.array([0, 0, 2, 2, 2], np.int32)
    s = C.Structure(cell, species, pos, rc, [calc])
    ref = oracle.B2Values(oracle.Neighbors(cell, species, pos, rc), *settings, cut)
    d = s.descriptors[0]
    for t in range(nos):
        assert rel_err(d.descriptor_force_dervs[t], ref.descriptor_force_dervs[t]) < 1e-10
        assert rel_err(d.descriptor_force_dots[t], ref.descriptor_force_dots[t]) < 1e-10
    kern = C.NormalizedDotProduct(1.7, power)
    sgp = C.SparseGP([kern], 0.01, 0.05, 0.005)
    atoms = [int(a) for t, m in enumerate(n_sparse) for a in d.atom_indices[t][:m]]
    sgp.add_specific_environments(s, atoms)
    cd = sgp.sparse_descriptors[0]
    assert cd.n_clusters_by_type == list(n_sparse)
    m = oracle.Model(1.7, power, cd.descriptors, cd.descriptor_norms, np.zeros(sum(n_sparse)))
    assert rel_err(kern.envs_struc(cd, d), m.envs_struc(ref)) < 1e-10
