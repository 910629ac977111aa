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
