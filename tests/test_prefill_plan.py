"""CPU: the prefill attention's plan (csrc/mg_prefill_plan.hpp, the header the
launcher compiles) keeps every tile's keys inside its parts.

A windowed call's middle tiles reach further than both end tiles: the first one
may start before the window fills, the last one may hold few rows. A plan sized
by the end tiles loses the middle rows' newest keys and lets the merge read
another tile's partials; the shapes below are some it went wrong at."""
import pathlib
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    exe = tmp_path_factory.mktemp("plan") / "prefill_plan_check"
    subprocess.run(["g++", "-std=c++17", "-O2", f"-I{ROOT / 'muse-glimmer-intel-serve_amd' / 'csrc'}",
                    str(ROOT / "tests" / "host" / "prefill_plan_check.cpp"), "-o", str(exe)], check=True)
    return exe


def run(exe, *args):
    return [int(v) for v in subprocess.run([str(exe), *map(str, args)], check=True, capture_output=True,
                                           text=True).stdout.split()]


@pytest.mark.parametrize("T,nq,nkv,pos0,window", (
    (57, 32, 2, 986, 1024),
    (129, 40, 8, 938, 1024),
    (1606, 1, 1, 0, 542),
))
def test_windowed_middle_tiles(checker, T, nq, nkv, pos0, window):
    assert run(checker, T, nq, nkv, pos0, window) == [1, 1, 1, 0]


def test_sweep(checker):
    plans, split, wsplit, bad = run(checker)
    assert split > 100000 and wsplit > 50000  # the sweep reaches what it checks
    assert bad == 0
