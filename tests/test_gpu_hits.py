"""The hit-parallel Metropolis kernel (sweep variants 16-19) against the oracle
and, bit for bit, against the site-wave kernel whose results it reproduces."""
import numpy as np
import pytest

import klft_amd as klft
import oracle as orc

pytestmark = pytest.mark.gpu

BETA = {1: 2.0, 2: 2.3, 3: 5.5}


def sweeps(monkeypatch, variant, nd, nc, dims, storage, nhits, U=None, n=3, law=None):
    monkeypatch.setenv("KLFT_VARIANT", variant)
    g = klft.GaugeField(nd, nc, dims, storage)
    g.upload(U) if U is not None else g.set_random_algebra(0.5, 7)
    if law:
        g.set_proposal(law)
    p = klft.MetropolisParams(nHits=nhits, beta=BETA[nc], delta=0.2, seed=123)
    counts = [klft.sweep_Metropolis(g, p, s, with_count=True)[1] for s in range(n)]
    out = g.download()
    g.close()
    return counts, out


# hits per link: fewer than a site's lanes, one round exactly (10), two rounds
# with a partly filled second one (13)
@pytest.mark.parametrize("nhits", [1, 10, 13])
@pytest.mark.parametrize("waves", [2, 4])
@pytest.mark.parametrize("nd,nc,dims", [(4, 3, (6, 4, 10, 4)), (4, 2, (6, 6, 4, 10)), (4, 1, (6, 6, 6, 6)),
                                        (3, 3, (10, 6, 12)), (3, 2, (4, 6, 10)), (2, 3, (10, 14)), (2, 1, (14, 10))])
def test_hits_match_oracle(monkeypatch, nd, nc, dims, waves, nhits):
    """FP64 decisions identical to the oracle's over three sweeps, links within
    1e-11, on lattices that leave the last block of a pass partly filled."""
    U = orc.random_algebra(nd, nc, dims, 0.4, 71)
    got, u = sweeps(monkeypatch, f"metropolis=17,hits_waves={waves}", nd, nc, dims, "f64", nhits, U)
    want = [orc.metropolis_sweep(U, nd, nc, dims, nhits, BETA[nc], 0.2, 123, s)[1] for s in range(3)]
    assert got == want
    np.testing.assert_allclose(u, U, rtol=0, atol=1e-11)


@pytest.mark.parametrize("storage", ["f64", "f32", "f32_rows"])
@pytest.mark.parametrize("order", [12, 13])
@pytest.mark.parametrize("nd,nc,dims", [(4, 3, (8, 6, 4, 10)), (4, 2, (6, 8, 4, 10)), (4, 1, (8, 8, 8, 8)),
                                        (3, 3, (10, 8, 12)), (2, 2, (6, 8))])
def test_hits_equal_site_waves(monkeypatch, nd, nc, dims, order, storage):
    """The same stream words, products and term order as the site-wave kernel:
    counts and links bit for bit (FP64 U(1): the last two bits of a link)."""
    a = sweeps(monkeypatch, f"metropolis={order}", nd, nc, dims, storage, 10)
    for waves in (2, 4):
        b = sweeps(monkeypatch, f"metropolis={order + 4},hits_waves={waves}", nd, nc, dims, storage, 10)
        assert a[0] == b[0]
        if nc == 1 and storage == "f64":
            np.testing.assert_allclose(a[1], b[1], rtol=0, atol=1e-14)
        else:
            assert np.array_equal(a[1], b[1])


@pytest.mark.parametrize("storage", ["f64", "f32"])
@pytest.mark.parametrize("nd,dims", [(4, (6, 6, 8, 4)), (2, (12, 10))])
def test_hits_symmetric_law(monkeypatch, nd, dims, storage):
    """The symmetric SU(3) proposal accepts most hits: many rounds per link."""
    a = sweeps(monkeypatch, "metropolis_pairs=0", nd, 3, dims, storage, 12, law="symmetric")
    U = orc.random_algebra(nd, 3, dims, 0.5, 7)
    if storage == "f64":
        want = [orc.metropolis_sweep_sym(U, nd, 3, dims, 12, BETA[3], 0.2, 123, s)[1] for s in range(3)]
        assert a[0] == want
        np.testing.assert_allclose(a[1], U, rtol=0, atol=1e-11)
    b = sweeps(monkeypatch, "hits_waves=2", nd, 3, dims, storage, 12, law="symmetric")
    assert a[0] == b[0] and np.array_equal(a[1], b[1])


@pytest.mark.parametrize("storage", ["f64", "f32_rows"])
@pytest.mark.parametrize("nd,nc,dims", [(4, 3, (8, 8, 8, 8)), (4, 1, (6, 6, 6, 6)), (3, 2, (8, 8, 8))])
def test_hits_runs_equal_single_sweeps(monkeypatch, nd, nc, dims, storage):
    """A run pairs independent passes, of one sweep and of consecutive ones:
    every sweep's rate and the links equal single sweeps without pairs, and the
    rates are those of the counts summed over the counter rows (runs of 3 and
    of 17 sweeps: the second's rows are longer than a line)."""
    p = klft.MetropolisParams(nHits=8, beta=BETA[nc], delta=0.2, seed=5)
    out = []
    for v in ("metropolis=17,metropolis_pairs=0", "metropolis=17"):
        monkeypatch.setenv("KLFT_VARIANT", v)
        g = klft.GaugeField(nd, nc, dims, storage).set_random_algebra(0.5, 2024)
        if "pairs" in v:
            rates = [klft.sweep_Metropolis(g, p, s) for s in range(20)]
        else:
            rates = [r for s0, n in ((0, 3), (3, 17)) for r in klft.metropolis_run(g, p, s0, n)]
        out.append((rates, g.download()))
        g.close()
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[0][1], out[1][1])


# one extent below and one above each limit of the default rule (sites of a
# pass per CU, 256 CUs): SU(3) 8 hits 81, SU(3) 1 hit 48, SU(2) 27, U(1) 20
@pytest.mark.parametrize("nc,nhits,dims", [(3, 8, (24, 24, 24, 24)), (3, 8, (24, 24, 24, 26)),
                                           (3, 1, (16, 24, 16, 32)), (3, 1, (16, 24, 16, 34)),
                                           (2, 6, (18, 18, 18, 18)), (2, 6, (18, 18, 18, 20)),
                                           (1, 6, (16, 16, 16, 20)), (1, 6, (16, 16, 16, 22))])
@pytest.mark.parametrize("storage", ["f64", "f32"])
def test_default_rule_keeps_results(monkeypatch, nc, nhits, dims, storage):
    """On both sides of a limit the default kernel gives the site-wave kernel's
    results."""
    a = sweeps(monkeypatch, "x=0", 4, nc, dims, storage, nhits, n=1)
    vh = np.prod(dims) // 16
    order = 13 if storage == "f64" or 2 * ((vh + 255) // 256) <= 256 else 12
    b = sweeps(monkeypatch, f"metropolis={order}", 4, nc, dims, storage, nhits, n=1)
    assert a[0] == b[0]
    if nc == 1 and storage == "f64":
        np.testing.assert_allclose(a[1], b[1], rtol=0, atol=1e-14)
    else:
        assert np.array_equal(a[1], b[1])
