"""Per-site plaquettes of many fields share the library's staging memory."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

import klft_amd as klft

pytestmark = pytest.mark.gpu


def sites(g, noalloc=False):
    """sum and sites; noalloc: the entry point with memory of its own, which
    copies straight into the caller's array"""
    out, ps = C.c_double(), np.full(g.volume, np.nan)
    fn = klft.lib.klft_plaquette_noalloc if noalloc else klft.lib.klft_plaquette
    assert fn(g.h, 0, C.byref(out), klft._dptr(ps)) == 0
    return out.value, ps


def test_fields_of_different_sizes_in_turn():
    """Growing, shrinking and growing again, across the size of a piece (2^17
    sites), and after every field was destroyed once."""
    for _ in range(2):
        gs = [klft.GaugeField(4, 1, d, "f64").set_random_algebra(0.5, i)
              for i, d in enumerate([(4, 4, 4, 4), (16, 16, 16, 16), (6, 4, 4, 4), (32, 16, 16, 18), (24, 16, 16, 16)])]
        for g in gs + gs[::-1]:
            a, b = sites(g), sites(g, noalloc=True)
            assert a[0] == b[0] and np.array_equal(a[1], b[1])
        for g in gs:
            g.close()


def test_array_beyond_what_is_kept():
    """9.4 million sites: 72 MiB, more than the 64 MiB that stay allocated."""
    g = klft.GaugeField(2, 1, (3072, 3072), "f32").set_random_algebra(0.5, 3)
    total, ps = sites(g)
    # the sites are FP32 values summed in FP64, in another order
    assert abs(ps.sum() - total) <= 1e-9 * g.volume
    assert np.isfinite(ps).all() and klft.GaugePlaquette(g, normalize=False) == total
    g.close()


def test_threads_take_turns():
    gs = [klft.GaugeField(4, 2, (8, 8, 8, 4 + 2 * i), "f64").set_random_algebra(0.5, i) for i in range(4)]
    want = [sites(g, noalloc=True) for g in gs]
    bad = []

    def work(i):
        for _ in range(20):
            a = sites(gs[i])
            if a[0] != want[i][0] or not np.array_equal(a[1], want[i][1]):
                bad.append(i)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
    for g in gs:
        g.close()


def test_first_call_of_a_field_allocates_nothing():
    """With one field measured, the first per-site call of each further field takes
    about as long as a later one (with pinned memory and an array of its own it took
    seven times as long)."""
    gs = [klft.GaugeField(4, 3, (16, 16, 16, 16), "f64").set_identity() for _ in range(25)]
    out, ps = C.c_double(), np.zeros(gs[0].volume)

    def timed(g):
        t = time.perf_counter()
        assert klft.lib.klft_plaquette(g.h, 1, C.byref(out), klft._dptr(ps)) == 0
        return time.perf_counter() - t

    for _ in range(3):
        timed(gs[0])
    first = np.median([timed(g) for g in gs[1:]])
    later = np.median([timed(g) for g in gs[1:]])
    assert first < 3 * later, (first, later)
    for g in gs:
        g.close()
