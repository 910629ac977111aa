"""Metropolis with a delta that is not a number or not finite: the proposals are
NaN, every hit is rejected and the call returns, in every sweep kernel."""
import numpy as np
import pytest

import oracle as orc
import klft_amd as klft

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("delta", [np.nan, np.inf])
@pytest.mark.parametrize("storage", ["f64", "f32", "f32_rows"])
@pytest.mark.parametrize("variant", [0, 7, 11, 12, 13, 16, 17])
def test_nonfinite_delta_is_rejected(monkeypatch, variant, storage, delta):
    monkeypatch.setenv("KLFT_VARIANT", f"metropolis={variant}")
    g = klft.GaugeField(4, 3, (4, 4, 6, 4), storage).set_random_algebra(0.4, 3)
    before = g.download()
    p = klft.MetropolisParams(nHits=3, beta=5.5, delta=delta, seed=5)
    assert klft.sweep_Metropolis(g, p, 0, with_count=True) == (0.0, 0)
    assert np.array_equal(g.download(), before)
    g.close()


@pytest.mark.parametrize("delta", [np.nan, np.inf])
@pytest.mark.parametrize("storage", ["f64", "f32"])
@pytest.mark.parametrize("variant", [0, 1, 2])
def test_nonfinite_delta_in_a_batch_is_rejected(monkeypatch, variant, storage, delta):
    monkeypatch.setenv("KLFT_VARIANT", f"batch={variant}")
    dims = (4, 4, 4, 6)
    U = orc.random_algebra(4, 3, dims, 0.4, 3)
    b = klft.Batch([(3, dims, 5.5), (3, dims, 6.0)], storage)
    for i in range(2):
        b.upload(i, U)
    before = b.download(1)
    assert np.array_equal(b.sweep(3, delta, 7, 0), [0.0, 0.0])
    assert np.array_equal(b.download(1), before)
    b.close()
    r = klft.PTBC(2, 3, dims, 5.5, 2, [0, 1, 2], [1.0, 0.5], storage)
    r.upload(0, U)
    before = r.download(0)
    r.step(3, delta, 7, 0)
    assert np.array_equal(r.download(0), before)
    r.close()


def test_delta_without_a_proposal_is_an_error():
    """SU(3) with the reference's law and a delta that no proposal can be drawn
    with: an error before any launch, the links unchanged.  Without hits or
    sweeps, with the symmetric law, or in U(1) and SU(2), the call runs."""
    dims = (4, 4, 4, 4)
    for storage in ("f64", "f32", "f32_rows"):
        g = klft.GaugeField(4, 3, dims, storage).set_random_algebra(0.4, 3)
        before = g.download()
        p = klft.MetropolisParams(nHits=2, beta=5.5, delta=0.0, seed=5)
        with pytest.raises(klft.KlftError, match="delta"):
            klft.sweep_Metropolis(g, p, 0)
        with pytest.raises(klft.KlftError, match="delta"):
            klft.metropolis_run(g, p, 0, 3)
        with pytest.raises(klft.KlftError, match="delta"):
            g.set_random_sun(0.0, 7)
        klft.metropolis_run(g, p, 0, 0)
        klft.sweep_Metropolis(g, klft.MetropolisParams(nHits=0, beta=5.5, delta=0.0, seed=5), 0)
        assert np.array_equal(g.download(), before)
        g.set_proposal("symmetric")
        assert klft.sweep_Metropolis(g, p, 0) > 0.99  # the identity, dS = 0 up to rounding
        g.close()
        b = klft.Batch([(1, dims, 2.0), (3, dims, 5.5)], storage)
        with pytest.raises(klft.KlftError, match="delta"):
            b.sweep(2, 0.0, 7, 0)
        with pytest.raises(klft.KlftError, match="delta"):
            b.run(2, 0.0, 7, 0, 2)
        b.run(2, 0.0, 7, 0, 0)
        b.close()
        r = klft.PTBC(2, 3, dims, 5.5, 2, [0, 1, 2], [1.0, 0.5], storage)
        with pytest.raises(klft.KlftError, match="delta"):
            r.step(2, 0.0, 7, 0)
        r.close()
        for nc in (1, 2):
            h = klft.GaugeField(4, nc, dims, storage).set_random_sun(0.0, 7)
            klft.sweep_Metropolis(h, p, 0)
            h.close()
