"""Wilson loops with the staple moved between lanes and through LDS, over column
lengths that fill, half fill, straddle and exceed a wave, against the FP64 oracle."""
import numpy as np
import pytest

import oracle as orc
import klft_amd as klft

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nt", [2, 6, 14, 24, 32, 62, 64, 66, 96, 260])
@pytest.mark.parametrize("nc,storage", [(1, "f64"), (2, "f64"), (3, "f64"), (1, "f32"), (3, "f32"), (2, "f32_rows"),
                                        (3, "f32_rows")])
@pytest.mark.parametrize("lanes", [0, 1])
def test_column_lengths_match_oracle(monkeypatch, nt, nc, storage, lanes):
    """Loops shorter than, as long as and longer than the extents, one extent
    given twice and out of order.  A site's loop is a product of at most 2 (L + T)
    <= 30 links and its trace: FP64 1e-12; FP32 30 links stored and multiplied with
    12 roundings of 2^-24 each at most, 2.2e-5 per colour."""
    monkeypatch.setenv("KLFT_VARIANT", f"wilson={lanes}")
    dims = (4, 6, nt)
    U = orc.random_algebra(3, nc, dims, 0.6, 23)
    g = klft.GaugeField(3, nc, dims, storage).upload(U)
    atol = 1e-12 if storage == "f64" else 2.2e-5 * nc
    pairs = [(3, 2), (1, 1), (5, 7), (0, 2), (2, 0), (8, 3), (3, 7)]
    for mu, nu in [(0, 2), (1, 2), (2, 0)]:
        ref, ref_ps = orc.wilson_mu_nu(U, 3, nc, dims, mu, nu, pairs, per_site=True)
        got, ps = klft.WilsonLoop_mu_nu(g, mu, nu, pairs, per_site=True)
        np.testing.assert_allclose(ps, ref_ps, rtol=0, atol=atol)
        np.testing.assert_allclose([w[4] for w in got], ref, rtol=0, atol=atol / nc)
    got = klft.WilsonLoop_temporal(g, pairs)
    np.testing.assert_allclose([w[2] for w in got], orc.wilson_temporal(U, 3, nc, dims, pairs), rtol=0, atol=atol / nc)
    g.close()
