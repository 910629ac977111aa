"""The leapfrog step and the force with one, two and all directions per thread,
with and without stores past the caches, against the FP64 oracle."""
import numpy as np
import pytest

import oracle as orc
import klft_amd as klft

pytestmark = pytest.mark.gpu

# sublattices of 84, 81, 150 and 135 sites: a part block after a full one, and
# extents of 2, where both neighbours are one site
SHAPES = [(4, (2, 6, 8, 14)), (4, (6, 6, 6, 6)), (3, (12, 10, 10)), (2, (30, 18))]


@pytest.mark.parametrize("nd,dims", SHAPES)
@pytest.mark.parametrize("nc,storage", [(1, "f64"), (2, "f64"), (3, "f64"), (1, "f32"), (2, "f32"), (3, "f32"),
                                        (2, "f32_rows"), (3, "f32_rows")])
def test_directions_per_thread_match_oracle(monkeypatch, nd, dims, nc, storage):
    """Two steps of the leapfrog and one momentum update.  FP64: 1e-12 as for the
    force.  FP32: an entry of U Sigma sums 2 (nd - 1) <= 6 terms of 3 products
    of at most 3 complex entries, each rounded at most 12 times, so F is off by
    at most 650 eps beta / Nc, P by that times tau plus 4 eps |P| <= 20 eps, and
    U by dtau times P's and its own product's and restoration's 30 eps: 2e-5 with
    beta / Nc = 1, tau = 0.25 and eps = 2^-24, links stored in FP32 included."""
    U = orc.random_algebra(nd, nc, dims, 0.6, 17)
    P = orc.refresh_momenta(nd, nc, dims, 5, 1)
    atol = 1e-12 if storage == "f64" else 2e-5
    beta, tau = float(nc), 0.25
    Ul, Pl = U.copy(), P.copy()
    orc.leapfrog(Ul, Pl, nd, nc, dims, beta, tau, 2)
    Pu = P.copy()
    orc.update_momentum(Pu, orc.force(U, nd, nc, dims, beta), nd, nc, dims, 0.125)
    for md, force in [(1, 4), (2, 5), (3, 6)]:
        for stream in (0, 1):
            monkeypatch.setenv("KLFT_VARIANT", f"md_step={md},force={force},md_stream={stream}")
            g = klft.GaugeField(nd, nc, dims, storage).upload(U)
            h = klft.HMC(g, beta=beta, tau=tau, nsteps=2, seed=5)
            h.set_momenta(P)
            h.update_momentum(0.125)
            np.testing.assert_allclose(h.momenta(), Pu, rtol=0, atol=atol)
            np.testing.assert_allclose(h.kinetic(), orc.kinetic(Pu, nd, nc, dims), rtol=0 if atol < 1e-9 else 1e-5,
                                       atol=1e-9)
            np.testing.assert_allclose(h.force(), orc.force(U, nd, nc, dims, beta), rtol=0, atol=4 * atol)
            h.set_momenta(P)
            h.integrate()
            np.testing.assert_allclose(h.momenta(), Pl, rtol=0, atol=atol)
            np.testing.assert_allclose(g.download(), Ul, rtol=0, atol=atol)
            h.close()
            g.close()
