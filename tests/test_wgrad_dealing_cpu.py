"""How tiles of weight gradients of uneven loads are dealt by depth (csrc/wgrad_deal.h), replayed on the host: every tile is dealt once, and the loads that
the kernel works out for both orders, to take the one whose largest is the smaller, are those that the workgroups get."""
import ctypes
import importlib
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "wgrad_deal.h"
using namespace amoe_deal;
// depths: of the experts; order: experts by depth, deepest first.  taken: by each tile's workgroup, or -1 - that if it was taken before;
// loads: by number and by depth as the kernel works them out
extern "C" void replay(int E, int per, const int* depths, const int* order, int* taken, int* loads)
{
    for (int i = 0; i < E * per; ++i) taken[i] = ALL;
    for (int i = 0; i < 2 * ALL; ++i) loads[i] = 0;
    Walk walk;
    auto by_number = [&](int w, int d) { loads[w] += d; };
    auto by_depth = [&](int w, int d) { loads[ALL + w] += d; };
    for (int k = 0; k < E; ++k) {
        const int e = order[k], d = depths[e];
        add_by_number(e, d, per, by_number);
        const Record w = walk.next(d, per), r = Record::of(w.word(), w.behind, w.fill);
        add_by_depth(r, d, per, by_depth);
        for (int my = 0; my < ALL; ++my)
            for (Turns t(r, my); t.at < per; t.next()) {
                int& who = taken[e * per + t.at];
                who = who == ALL ? my : -1 - my;
            }
    }
    const int whole = E * per / ALL * ALL;
    for (int i = 0; i < E * per - whole; ++i) {
        const int d = depths[(whole + i) / per];
        add_arc(i, 1, -d, by_number);
        add_arc(last_of(i), 1, d, by_number);
    }
    for (int s = 0; s < 2; ++s)
        for (int i = 1; i < ALL; ++i) loads[s * ALL + i] += loads[s * ALL + i - 1];
}
"""


@pytest.fixture(scope="module")
def replay(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("deal")
    (d / "replay.cpp").write_text(SOURCE)
    subprocess.run([gxx, "-std=c++17", "-O2", "-shared", "-fPIC", "-Wall", "-Werror", "-I", os.path.join(ROOT, "arctictraining_amd", "csrc"),
                    str(d / "replay.cpp"), "-o", str(d / "replay.so")], check=True)
    lib = ctypes.CDLL(str(d / "replay.so"))

    def run(rows, per):
        depths = np.maximum(3, -(-np.asarray(rows, dtype=np.int64) // 64)).astype(np.int32) + 3
        E = len(depths)
        order = np.lexsort((np.arange(E), -depths)).astype(np.int32)
        taken, loads = np.empty(E * per, np.int32), np.empty((2, 256), np.int32)
        ptr = lambda a: a.ctypes.data_as(ctypes.c_void_p)  # noqa: E731
        lib.replay(E, per, ptr(depths), ptr(order), ptr(taken), ptr(loads))
        assert taken.min() >= 0 and taken.max() < 256   # every tile by one workgroup
        of_tile = np.repeat(depths, per).astype(np.int64)
        assert np.array_equal(np.bincount(taken, weights=of_tile, minlength=256).astype(np.int64), loads[1])
        v = np.arange(E * per)
        whole = E * per // 256 * 256
        last = v - whole
        who = np.where(v < whole, v % 256, (last & 7) * 32 + (last >> 3))   # an eighth of the last round to each of 8 dies
        assert np.array_equal(np.bincount(who, weights=of_tile, minlength=256).astype(np.int64), loads[0])
        uneven = depths.max() * E > 2 * depths.sum()
        return loads.max(axis=1), loads.sum() / 512, uneven

    return run


def _uneven(rng, E, R, kind):
    if kind == 0:
        p = np.arange(1, E + 1, dtype=float) ** -rng.uniform(0.6, 2.0)
    elif kind == 1:   # a few with half
        n = max(1, E // 16)
        p = np.r_[np.full(n, 0.5 / n), np.full(E - n, 0.5 / (E - n))]
    else:
        p = rng.lognormal(0, rng.uniform(0.5, 2.0), E)
    return rng.multinomial(R, rng.permutation(p / p.sum()) if rng.random() < 0.5 else p / p.sum())


@pytest.mark.parametrize("per", [1, 3, 7, 48, 88, 100, 128, 200, 250, 251, 252, 253, 254, 255, 256, 257, 300, 511, 513, 1792])
def test_dealt_once_and_loads_as_compared(replay, per):
    rng = np.random.default_rng(per)
    chosen = refused = 0
    for _ in range(60):
        E = int(rng.choice([2, 3, 5, 8, 13, 32, 64, 67, 128, 130, 509, 512]))
        if E * per > 300000 or E * per <= 256:
            continue
        (number, depth), mean, uneven = replay(_uneven(rng, E, int(E * rng.integers(704, 8000)), int(rng.integers(3))), per)
        assert mean <= depth and mean <= number
        if uneven:
            chosen += depth < number
            refused += depth >= number
    assert chosen + refused >= 5


def test_loads_that_by_depth_made_worse(replay):
    """8 experts of 253 and 250 tiles, Zipf 1.2: by number within 1.02 and 1.03 of the mean"""
    p = np.arange(1, 9, dtype=float) ** -1.2
    rows = np.floor(32768 * p / p.sum()).astype(int)
    for per in (253, 250):
        (number, depth), mean, uneven = replay(rows, per)
        assert uneven and depth > number and number <= 1.03 * mean   # by number


def test_a_sixteenth_with_half_of_the_rows(replay):
    rows = [16384] * 4 + [1092] * 60   # 64 experts, 2048 x 1408: 88 tiles of gate_up's gradient
    (number, depth), mean, uneven = replay(rows, 88)
    assert uneven and depth < number and depth <= 1.02 * mean < 1.15 * mean <= number


@pytest.mark.parametrize("module", ["test_gpu_wgrad_dealing", "test_gpu_wgrad_dealing_wide"])
def test_gpu_cases_are_dealt_by_depth(replay, module):
    """(those that are meant to be: the GPU tests see results, not the order)"""
    for name, (rows, M, N) in importlib.import_module(module).CASES.items():
        per = -(-M // 256) * -(-N // 256)
        (number, depth), mean, uneven = replay(rows, per)
        depths = sum(max(3, -(-r // 64)) + 3 for r in rows)
        assert sum(rows) >= 704 * len(rows) and per * len(rows) > 256 and depths * per >= 1024 * len(rows), name
        assert (uneven and depth < number) == (name != "too_even"), (name, number, depth, mean)
