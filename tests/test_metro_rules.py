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
