"""The sweep kernels of the symmetric SU(3) proposal: site waves (variants 14, 15)
and hits in parallel (18, 19), each asked for by its number or by that of the
reference law's variant."""
import numpy as np
import pytest

import klft_amd as klft

pytestmark = pytest.mark.gpu


def sweeps(monkeypatch, variant, dims, storage, nhits=6, n=3):
    monkeypatch.setenv("KLFT_VARIANT", variant)
    g = klft.GaugeField(len(dims), 3, dims, storage).set_random_algebra(0.5, 7).set_proposal("symmetric")
    p = klft.MetropolisParams(nHits=nhits, beta=5.5, delta=0.2, seed=123)
    counts = [klft.sweep_Metropolis(g, p, s, with_count=True)[1] for s in range(n)]
    out = g.download()
    g.close()
    return counts, out


@pytest.mark.parametrize("storage", ["f64", "f32", "f32_rows"])
@pytest.mark.parametrize("order", [12, 13])
# part blocks of both kernels; 2D, where no two passes pair
@pytest.mark.parametrize("dims", [(8, 6, 4, 10), (10, 8, 12), (12, 10), (24, 12, 10, 12)])
def test_symmetric_hits_equal_site_waves(monkeypatch, dims, order, storage):
    """The same stream words, products and term order: counts and links bit for
    bit, and a variant's own number runs the same kernel as its counterpart's."""
    a = sweeps(monkeypatch, f"metropolis={order}", dims, storage)
    for v in (order + 2, order + 4, order + 6):
        b = sweeps(monkeypatch, f"metropolis={v}", dims, storage)
        assert a[0] == b[0] and np.array_equal(a[1], b[1]), v


def test_symmetric_variant_is_the_one_asked_for(monkeypatch):
    """FP64 at 32^4: the passes of the site waves (one block per CU) do not pair,
    those of the hit-parallel kernel always do."""
    klft.profile(True)
    try:
        for v, pairs in ((13, 0), (15, 0), (17, 5), (19, 5)):
            sweeps(monkeypatch, f"metropolis={v}", (32, 32, 32, 32), "f64", nhits=1, n=1)
            assert klft.profile_read("metropolis_pass_pair")[1] == pairs
    finally:
        klft.profile(False)
