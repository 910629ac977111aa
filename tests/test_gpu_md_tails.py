"""The leapfrog step and the force on sublattices whose last block holds few
sites, where the lanes beyond them repeat the last site."""
import numpy as np
import pytest

import oracle as orc
import klft_amd as klft

pytestmark = pytest.mark.gpu


# sublattices of 1, 16, 65 and 80 sites in 4D, of 12 in 3D and of 65 in 2D
@pytest.mark.parametrize("dims", [(2, 2, 2, 2), (4, 4, 4, 4), (2, 2, 10, 26), (4, 4, 10, 8), (4, 4, 6), (10, 26)])
@pytest.mark.parametrize("nc,storage", [(1, "f64"), (2, "f32"), (3, "f64"), (3, "f32"), (3, "f32_rows")])
def test_short_blocks_match_oracle(monkeypatch, dims, nc, storage):
    """Two leapfrog steps and a momentum update with two and all directions per
    thread.  Tolerances as in test_gpu_md.py: 1e-12 in FP64, 2e-5 in FP32 (beta /
    Nc = 1, tau = 0.25)."""
    nd = len(dims)
    U = orc.random_algebra(nd, nc, dims, 0.6, 17)
    P = orc.refresh_momenta(nd, nc, dims, 5, 1)
    atol = 1e-12 if storage == "f64" else 2e-5
    beta, tau = float(nc), 0.25
    Ul, Pl, Pu = U.copy(), P.copy(), P.copy()
    orc.leapfrog(Ul, Pl, nd, nc, dims, beta, tau, 2)
    orc.update_momentum(Pu, orc.force(U, nd, nc, dims, beta), nd, nc, dims, 0.125)
    for md, force in [(2, 5), (3, 6)]:
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


@pytest.mark.parametrize("storage", ["f64", "f32", "f32_rows"])
def test_kinetic_sum_counts_each_site_once(monkeypatch, storage):
    """The trajectory's closing force launch sums the kinetic energy: the energy
    change of a short one is that of the momenta it leaves."""
    dims = (2, 2, 10, 26)
    monkeypatch.setenv("KLFT_VARIANT", "md_step=3,force=6")
    g = klft.GaugeField(4, 3, dims, storage).set_random_algebra(0.4, 7)
    h = klft.HMC(g, beta=5.5, tau=0.02, nsteps=2, seed=3)
    h.refresh_momenta(4)
    before = orc.kinetic(h.momenta(), 4, 3, dims) + klft.gauge_action(g, 5.5)
    dH, accepted = h.trajectory(4)
    after = orc.kinetic(h.momenta(), 4, 3, dims) + klft.gauge_action(g, 5.5)
    assert accepted
    # FP32: the links are rounded at every step and the action of 6240 plaquettes
    # is a few thousand
    np.testing.assert_allclose(dH, after - before, rtol=0, atol=1e-8 if storage == "f64" else 0.05)
    g.close()


@pytest.mark.parametrize("storage", ["f64", "f32", "f32_rows"])
def test_short_blocks_take_no_longer(monkeypatch, storage):
    """SU(3) 6x6x8x8 has blocks of 16 sites among its 48, 8^4 64 blocks of 64: a step
    of the smaller lattice is not the longer one (it took 1.4 to 1.8 times as
    long)."""
    monkeypatch.setenv("KLFT_VARIANT", "md_step=3")
    t = []
    for dims in ((6, 6, 8, 8), (8, 8, 8, 8)):
        g = klft.GaugeField(4, 3, dims, storage).set_random_algebra(0.4, 7)
        h = klft.HMC(g, beta=6.0, tau=0.05, nsteps=30, seed=3)
        h.refresh_momenta(0)
        h.integrate()
        klft.profile(True)
        one = []
        for _ in range(7):
            h.integrate()
            ms, n = klft.profile_read("md_step")
            one.append(ms / n)
        klft.profile(False)
        t.append(np.median(one))
        h.close()
        g.close()
    assert t[0] < 1.25 * t[1], t


def test_small_lattices_take_a_thread_per_link(monkeypatch):
    """The default rule in SU(3), below, inside and above 17 to 64 sites of a
    sublattice: the step's results are those of the variant it stands for."""
    for dims, md, force in (((4, 4, 4, 4), 3, 6), ((4, 4, 6, 4), 1, 4), ((4, 4, 8, 8), 1, 4), ((4, 4, 10, 8), 3, 6)):
        out = []
        for v in ("x=0", f"md_step={md},force={force}"):
            monkeypatch.setenv("KLFT_VARIANT", v)
            g = klft.GaugeField(4, 3, dims, "f64").set_random_algebra(0.4, 7)
            h = klft.HMC(g, beta=6.0, tau=0.2, nsteps=4, seed=3)
            h.refresh_momenta(0)
            h.integrate()
            out.append((g.download(), h.momenta()))
            h.close()
            g.close()
        assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
