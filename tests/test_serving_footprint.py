"""The bytes by which a server admits a request cover the buffers of its batch."""
import pytest

from flare_amd.serving import footprint_bytes


@pytest.mark.parametrize("esz", [4, 8])
@pytest.mark.parametrize("nd,n_rad_h,sparse", [(180, 200, 2000), (2100, 1176, 500), (20, 16, 16)])
def test_footprint_covers_buffers(esz, nd, n_rad_h, sparse):
    n, nnb = 5000, 5000 * 40
    up = lambda a, b: -(-a // b)
    rows = 2 * esz * nd + 2 * esz * n_rad_h  # B and G, c and u
    k = 8 * 16 * up(sparse, 16)
    variance = 8 * 2 * up(sparse, 64)
    if esz == 8:
        model = k + k + 8 * up(sparse, 16) + variance  # k, w and the energy partials
    else:
        model = k + 4 * 32 * up(sparse, 32) + 8 * up(sparse, 64) + variance + 5 * nd
    lists = 4 + 4 + 32 + 4 * 4 + 3 * esz  # neighbours, bonds (two lists and two of the build), forces
    assert footprint_bytes(n, nnb, nd, n_rad_h, sparse, esz) >= n * (rows + model) + nnb * lists
