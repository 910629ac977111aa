"""The sweep's rules (metro_rules.hpp) on the CPU, compiled by the host compiler
from the header that the library's kernels and host code use."""
import subprocess
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    exe = tmp_path_factory.mktemp("rules") / "metro_rules"
    subprocess.run(["g++", "-O1", "-std=c++17", f"-I{ROOT / 'klft_amd' / 'csrc'}", "-o", str(exe),
                    str(ROOT / "tests" / "helpers" / "metro_rules.cpp")], check=True)

    def call(*args):
        out = subprocess.run([str(exe), *map(str, args)], capture_output=True, text=True, check=True).stdout
        return [[float(v) for v in line.split()] for line in out.splitlines()]
    return call


def test_row_is_redrawn_as_the_reference_does(rules):
    """randSUN<3> draws a row again unless 1 != 1 + norm (SUN.hpp:198-233): the
    rule on the squared norm takes the same decision, at its edge, for subnormal,
    infinite and NaN values, and over the whole range of magnitudes."""
    edge = 2.0 ** -106
    n2 = [0.0, 5e-324, 1e-300, np.nextafter(edge, 0), edge, np.nextafter(edge, 1), edge * (1 + 2.0 ** -51),
          edge * (1 + 2.0 ** -50), 1e-30, 0.06, 1.0, 6.0, 1e300, np.inf, np.nan]
    n2 += list(10.0 ** np.random.default_rng(5).uniform(-320, 300, 500))
    n2 += list(edge * (1 + np.random.default_rng(6).uniform(-4, 4, 200) * 2.0 ** -52))
    want = [not (1.0 != 1.0 + np.sqrt(v)) for v in np.array(n2)]
    got = [bool(v[0]) for v in rules("row_redrawn", *[float(v).hex() for v in n2])]
    assert got == want


@pytest.mark.parametrize("delta", ["nan", "inf", "-inf", "0.1", "1e-12", "1e100"])
def test_drawing_a_row_ends(rules, delta):
    """The loop that draws a row is left after one draw, also for a delta that is
    not finite."""
    for seed in range(20):
        assert rules("rows_drawn", delta, seed, 50) == [[1, 0]]


@pytest.mark.parametrize("fp64,smallest,largest", [(1, 2.0 ** -54, 2.0 ** 513), (0, 2.0 ** -25, 2.0 ** 65)])
def test_delta_without_a_proposal(rules, fp64, smallest, largest):
    """Only a delta whose rows are next to never kept is refused: zero, below half
    the smallest norm, above twice the largest (FP32 links: as a float).  One at the
    limits keeps a row within some thousand draws."""
    keep = [smallest, -smallest, largest, 0.1, 1.0, 1e-6, np.nan, np.inf, -np.inf] + ([] if fp64 else [1e300])
    drop = [0.0, -0.0, 5e-324, smallest * (1 - 2.0 ** -22), largest * (1 + 2.0 ** -22), -2 * largest]
    got = [bool(v[0]) for v in rules("rows_kept", fp64, *[float(d).hex() for d in keep + drop])]
    assert got == [True] * len(keep) + [False] * len(drop)
    if fp64:
        for d in (smallest, -smallest):
            assert rules("rows_drawn", d.hex(), 3, 20000)[0][1] == 0
        assert rules("rows_drawn", "0", 3, 1000) == [[1000, 1]]


# sites of a pass on 256 CUs: 16^4, 18^4, 20^4, 22^4, 24^4
VH = {L: L ** 4 // 16 for L in (16, 18, 20, 22, 24, 26)}


@pytest.mark.parametrize("nc,nhits,beta,law,largest", [
    # SU(3): the limit falls with the acceptance
    (3, 10, 6.0, 0, 24), (3, 10, 5.0, 0, 22), (3, 10, 4.0, 0, 20), (3, 10, 2.5, 0, 16), (3, 10, 0.5, 0, 16),
    (3, 10, 6.0, 1, 18), (3, 4, 6.0, 0, 20), (3, 4, 4.0, 0, 18), (3, 4, 0.5, 0, 16), (3, 4, 6.0, 1, 18),
    (3, 1, 6.0, 0, 20), (3, 1, 2.5, 0, 16), (3, 1, 6.0, 1, 16), (3, 10, "nan", 0, 16), (3, 10, -5.0, 0, 16),
    # SU(2), U(1): the same limit for every beta
    (2, 10, 2.3, 0, 18), (2, 10, 0.1, 1, 18), (1, 10, 2.0, 0, 16), (1, 4, 0.1, 0, 20)])
def test_hits_in_parallel_up_to_the_measured_size(rules, nc, nhits, beta, law, largest):
    """The largest 4D lattice whose sweep takes the hit-parallel kernel, by group,
    hits, beta and law.  Smaller ones always do, but for short hit chains in 2D."""
    for L, vh in VH.items():
        assert bool(rules("hits_in_parallel", 4, nc, vh, 256, nhits, beta, law)[0][0]) == (L <= largest), L
    assert rules("hits_in_parallel", 4, nc, 14 ** 4 // 16, 256, nhits, beta, law) == [[1]]
    assert rules("hits_in_parallel", 2, nc, 256, 256, 3, beta, law) == [[0]]
    assert rules("hits_in_parallel", 2, nc, 256, 256, 4, beta, law) == [[1]]
