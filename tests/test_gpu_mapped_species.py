"""The mapped potential over its launches for all species: one, eight (one
launch) and nine species (two), some without atoms, results of up to 256 KB
(read back by one kernel) and larger ones. Against the oracle."""
import numpy as np
import pytest

from helpers import random_cell, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("power", [1, 2])
@pytest.mark.parametrize("nos,n", [(1, 1), (8, 40), (9, 41), (2, 8191), (2, 8300)])
def test_mapped_species(oracle, tmp_path, nos, n, power):
    from flare_amd import _C_flare as C
    from flare_amd.mapping import MappedPotential
    rc, N, L = 3.2, 2, 1
    cell, species, pos = random_cell(n, 90 + nos, nos=nos, scale=3.0 if n == 1 else 2.3 * n ** (1 / 3),
                                     skew=0.1)
    species[species == 1] = 0 if n < 100 else 1  # a species without atoms
    nr = nos * N
    d = nr * (nr + 1) // 2 * (L + 1)
    size = d if power == 1 else d * (d + 1) // 2
    beta = np.random.default_rng(nos).normal(size=(nos, size))
    lines = ["DATE: x CONTRIBUTOR: y", "%d NormalizedDotProduct" % power, "chebyshev",
             "%d %d %d %d" % (nos, N, L, size), "quadratic"]
    lines.append(" ".join(["%.17g" % rc] * nos * nos))
    for row in beta:
        lines += [" ".join("%.17g" % v for v in row[k:k + 5]) for k in range(0, size, 5)]
    text = "\n".join(lines) + "\n"
    path = tmp_path / "lmp.flare"
    path.write_text(text)
    mp = MappedPotential(str(path))
    e, F, vir = mp.compute(cell, species, pos)
    e_ref, F_ref, vir_ref = oracle.pair_flare(text, oracle.Neighbors(cell, species, pos, rc, "cells"))
    assert rel_err(e, e_ref) < 1e-10
    assert rel_err(F, F_ref) < 1e-10
    assert rel_err(vir, vir_ref) < 1e-10
