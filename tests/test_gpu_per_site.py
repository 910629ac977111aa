"""Per-site plaquettes through the pinned pieces: fewer than one, exactly one, two
and a remainder, and two and a whole one of 2^17 values each."""
import ctypes as C

import numpy as np
import pytest

import klft_amd as klft

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(4, 4, 2, 2), (32, 16, 16, 16), (24, 24, 24, 20), (48, 32, 16, 16)])
def test_per_site_equals_plain_copy(dims):
    """The entry point without device allocations copies straight into the
    caller's array and runs the same kernel: the same bytes, on a first call, on a
    second with other links, and after loops used the workspace."""
    g = klft.GaugeField(4, 1, dims, "f64")
    for seed in (1, 2):
        g.set_random_algebra(0.5, seed)
        want, out = np.full(g.volume, np.nan), C.c_double()
        assert klft.lib.klft_plaquette_noalloc(g.h, 1, C.byref(out), klft._dptr(want)) == 0
        got, ps = klft.GaugePlaquette(g, per_site=True)
        assert np.array_equal(ps, want) and got == out.value
        klft.WilsonLoop_temporal(g, [(1, 1), (2, 2)])
    g.close()
