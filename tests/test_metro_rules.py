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
