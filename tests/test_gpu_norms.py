"""The FP64 inverse norms behind restoreSUN (v_rsq_f64 and one third-order
step, sqrt and division outside 2^-900 .. 2^900) against sqrt and division."""
import numpy as np
import pytest

import klft_amd as klft

pytestmark = pytest.mark.gpu


def restored(u):
    """Real and imaginary parts of restoreSUN<1> / <2> of a matrix, in numpy
    (SUN.hpp:256-300)."""
    with np.errstate(all="ignore"):
        n = np.sqrt(np.sum(u[0].real ** 2 + u[0].imag ** 2))
        return u.real / n, u.imag / n


@pytest.mark.parametrize("nc", [1, 2])
@pytest.mark.parametrize("z", [1.0, 1 + 2j, 3e-130 - 1e-130j, 2e130j, -7e-137 + 1e-137j, 5e-324, 3e-162 + 1e-162j,
                               1e-200, 0.0, 1e150 + 1e150j, 1e160, -1e300j])
def test_reunitarize_constant_links(nc, z):
    """Magnitudes inside the fast range, at its edges, and where the squared
    norm is subnormal, zero or infinite.  Inside: one rounding of n2, inv_sqrt
    within 1 ulp and the product's half, against sqrt's and the division's
    halves: 3 ulp.  Outside: the same infinities, zeros and NaNs."""
    g = klft.GaugeField(2, nc, (2, 2), "f64").set_constant(z)
    g.reunitarize()
    want = restored(np.full((nc, nc), complex(z)))
    got = g.download().reshape(-1, nc, nc)
    for a, b in zip((got.real, got.imag), want):
        b = np.broadcast_to(b, a.shape)
        assert np.array_equal(np.isnan(a), np.isnan(b))
        fine = np.isfinite(b)
        assert np.array_equal(a[~fine & ~np.isnan(b)], b[~fine & ~np.isnan(b)])
        # a subnormal squared norm has few digits: both sides round it alike
        np.testing.assert_allclose(a[fine], b[fine], rtol=3 * 2.0 ** -52, atol=0)


def test_reunitarized_random_links_are_unit():
    """SU(3) links of general complex entries: both rows of unit norm and the
    third their cross product, to a few ulp."""
    g = klft.GaugeField(4, 3, (4, 4, 6, 4), "f64").set_random_complex(5).reunitarize()
    u = g.download().reshape(-1, 3, 3)
    np.testing.assert_allclose(np.sum(np.abs(u[:, 0]) ** 2, axis=1), 1.0, rtol=0, atol=8 * 2.0 ** -52)
    np.testing.assert_allclose(np.cross(u[:, 2], u[:, 0]).conj(), u[:, 1], rtol=0, atol=8 * 2.0 ** -52)
