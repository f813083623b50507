"""The build of a structure (neighbour list, species rows, bond lists) at the
edges of its launches: 1,024 atoms per row block, 8,192 values per one-block
scan, cutoffs by value up to four species, and host arrays staged or not."""
import numpy as np
import pytest

from helpers import random_cell

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nos", [1, 3, 5])
@pytest.mark.parametrize("n", [1, 64, 1023, 1024, 1025, 8192, 8193, 10000])
def test_lists_and_rows(oracle, n, nos):
    from flare_amd import _C_flare as C
    rc = 3.0
    cell, species, pos = random_cell(n, 80 + nos, nos=nos, scale=4.0 if n == 1 else 2.4 * n ** (1 / 3),
                                     skew=0.1)
    # Pair cutoffs below the neighbour cutoff for all but the last species.
    cut = np.full((nos, nos), 2.7)
    cut[-1, -1] = rc
    calc = C.B2("chebyshev", "quadratic", [0.0, rc], [], [nos, 1, 0], cut)
    s = C.Structure(cell, species, pos, rc, [calc])
    ref = oracle.Neighbors(cell, species, pos, rc, "cells")
    assert s.n_neighbors == ref.n_neighbors
    assert np.array_equal(s.neighbor_count, ref.neighbor_count)
    assert np.array_equal(s.structure_indices, ref.structure_indices)
    assert np.array_equal(s.relative_positions, ref.relative_positions)
    d = s.descriptors[0]
    order = np.argsort(species, kind="stable")
    assert d.n_clusters_by_type == [int((species == t).sum()) for t in range(nos)]
    assert np.array_equal(np.concatenate(d.atom_indices), order)
    centre = np.repeat(species, ref.neighbor_count)
    r = ref.relative_positions[:, 0]
    keep = r <= cut[centre, species[ref.structure_indices]]
    assert d.n_neighbors_by_type == [int(keep[centre == t].sum()) for t in range(nos)]
    per_atom = np.add.reduceat(np.r_[keep, 0], np.r_[0, np.cumsum(ref.neighbor_count)[:-1]]) * (ref.neighbor_count > 0)
    assert np.array_equal(np.concatenate(d.neighbor_counts), per_atom[order])


@pytest.mark.parametrize("n", [2, 2047, 2048, 2049, 8191])
def test_lists_and_rows_small(oracle, n):
    """At the edges of the builds in one workgroup (2,048 atoms; 8,192)."""
    test_lists_and_rows(oracle, n, 3)


@pytest.mark.parametrize("side", [161, 162, 211])
def test_lists_in_a_large_cell(oracle, side):
    """Pairs of atoms in cells of 4.17, 4.25 and 9.4 million bins: from 4,096 blocks
    of 1,024 on the scan of the bins scans the blocks' totals first."""
    from flare_amd import _C_flare as C
    rng = np.random.default_rng(side)
    cell = np.eye(3) * (side * (1 + 1e-6))
    one = rng.uniform(0, side, (150, 3))
    one[0], one[1] = 0.1, side - 0.05  # the first and the last bin
    pos = np.concatenate([one, one + rng.uniform(-0.6, 0.6, one.shape)])
    species = np.zeros(len(pos), np.int32)
    s = C.Structure(cell, species, pos, 0.999, [])
    ref = oracle.Neighbors(cell, species, pos, 0.999, "literal")
    assert s.n_neighbors == ref.n_neighbors > 100
    assert np.array_equal(s.neighbor_count, ref.neighbor_count)
    assert np.array_equal(s.structure_indices, ref.structure_indices)
    assert np.array_equal(s.relative_positions, ref.relative_positions)
