"""The descriptor kernel over its waves per atom (one, two and four), rows of
one, three and more tiles of radial functions, staged in LDS or too long for
it, and one to three chunks of bonds: FP64 rows against the oracle, the chosen
form's energies, forces, stress and variances too."""
import numpy as np
import pytest

from helpers import random_cell, rel_err

pytestmark = pytest.mark.gpu

# (species, radial functions, l_max)
SETTINGS = [(1, 4, 2), (3, 7, 2), (5, 7, 0),  # one wave, up to 16, 32 and 35 functions
            (2, 8, 4), (5, 7, 1),             # two waves
            (2, 8, 6), (3, 8, 6), (4, 12, 3),  # four waves
            (8, 12, 4)]                       # 186 KB row


@pytest.mark.parametrize("settings", SETTINGS)
@pytest.mark.parametrize("n,rc", [(1, 4.0), (37, 4.5), (50, 6.5)])
def test_descriptor_rows(oracle, settings, n, rc):
    from flare_amd import _C_flare as C
    nos = settings[0]
    cut = np.full((nos, nos), rc)
    calc = C.B2("chebyshev", "quadratic", [0.0, rc], [], list(settings), cut)
    system = random_cell(n, 60 + n, nos=nos, scale=3.2 if n == 1 else 2.2 * n ** (1 / 3), skew=0.2)
    s = C.Structure(*system, rc, [calc])
    d = s.descriptors[0]
    ref = oracle.B2Values(oracle.Neighbors(*system, rc), *settings, cut)
    for t in range(nos):
        assert rel_err(d.descriptors[t], ref.descriptors[t]) < 1e-10
        assert rel_err(d.descriptor_norms[t], ref.descriptor_norms[t]) < 1e-10

    sgp = C.SparseGP([C.NormalizedDotProduct(1.5, 2.0)], 0.01, 0.05, 0.005)
    sgp.add_specific_environments(s, list(range(min(n, 20))))
    sgp.update_L_inverse()
    sgp.set_alpha(np.random.default_rng(5).uniform(0.1, 1.0, size=sgp.n_sparse))
    cd = sgp.sparse_descriptors[0]
    model = oracle.Model(1.5, 2.0, cd.descriptors, cd.descriptor_norms, sgp.alpha, L_inv=sgp.L_inv)
    mean, var = model.predict(ref, "local")
    p = C.Structure(*system, rc, [calc], form=C.FORM_CHOSEN)
    sgp.predict_local_uncertainties(p)
    # Slices carry the rows to 2^-34 of the largest element; the adjoint of
    # the forces is FP32 with split-BF16 products (2^-16 per product).
    m = p.mean_efs
    assert abs(m[0] - mean[0]) < 1e-6 * abs(mean[0])
    scale = max(np.max(np.abs(mean[1:])), 1e-3 * abs(mean[0]))
    assert np.max(np.abs(m[1:] - mean[1:])) < 1e-3 * scale
    assert np.max(np.abs(p.local_uncertainties[0] - var)) < 1e-3 * 1.5 ** 2


@pytest.mark.parametrize("settings", [(3, 10, 6), (2, 9, 4), (1, 5, 0), (3, 10, 5), (2, 14, 4)])
def test_projection_rows(oracle, settings):
    """The adjoint's rows in one pass: 3255 values (single elements), 855 and 15
    (unaligned vectors), 2790 and 2030 (odd counts of vectors)."""
    test_descriptor_rows(oracle, settings, 37, 4.5)


# One (l_max 2), three (5), four (7) and eight tiles of harmonics (8 to 10) on
# one, two and four waves; one wave with eight and ten atoms on a CU.
@pytest.mark.parametrize("settings", [(1, 5, 2), (1, 1, 5), (1, 4, 5), (2, 9, 5), (2, 6, 7), (1, 3, 8),
                                      (1, 4, 9), (2, 5, 10), (2, 8, 3), (1, 8, 4)])
@pytest.mark.parametrize("n,rc", [(1, 4.0), (50, 6.5)])
def test_tiles_of_harmonics(oracle, settings, n, rc):
    test_descriptor_rows(oracle, settings, n, rc)
