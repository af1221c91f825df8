"""The sorting networks that order the nearest entries of a column's list and the walk over them (``csrc/gd_order.h``), compiled for the host; and columns with
lists of one to six such windows, drawn with a lane a column, against the CPU oracle."""

from __future__ import annotations

import ctypes as C
import os
import subprocess

import numpy as np
import pytest
import torch

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "env-gradoom-turbo-torch_amd", "csrc")

DRIVER = r"""
#include "gd_order.h"
extern "C" void order_numbers(double *v) { order_up(*reinterpret_cast<double (*)[16]>(v)); }
extern "C" void lowest_of(double *v, double *other) {
    order_merge_lowest(*reinterpret_cast<double (*)[16]>(v), *reinterpret_cast<double (*)[16]>(other));
}
// a walk over distances: which rows were looked at as there, where `from` went, whether it ended
struct Entry { float dist; int at; };
extern "C" int walk(const float *rows, int count, int *from, int held, float passed, float limit, int advance, int *looked) {
    auto row = [&](int k) { if (k >= count) __builtin_trap(); return Entry{rows[k], k}; };
    auto look = [&](const Entry &e, bool there) { looked[e.at] += there ? 1 : 0; };
    auto enough = [&]() { return limit; };
    return advance ? window_walk<true>(*from, held, passed, row, look, enough) : window_walk<false>(*from, held, passed, row, look, enough);
}
"""


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    path = str(tmp_path_factory.mktemp("order") / "liborder.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-Wno-unknown-pragmas", "-I", CSRC, "-x", "c++", "-o", path, "-"], input=DRIVER, text=True, check=True)
    return C.CDLL(path)


def test_the_networks_order_numbers(library):
    pointer = lambda values: values.ctypes.data_as(C.c_void_p)  # noqa: E731
    for bits in range(1 << 16):              # zeros and ones: what a network orders of these it orders of all numbers
        row = np.array([bits >> k & 1 for k in range(16)], dtype=np.float64)
        library.order_numbers(pointer(row))
        assert np.all(np.diff(row) >= 0.0)
    for ones in np.ndindex(17, 17):          # all pairs of ordered runs of them
        runs = [np.concatenate([np.zeros(16 - n), np.ones(n)]) for n in ones]
        lowest = np.sort(np.concatenate(runs))[:16]
        library.lowest_of(pointer(runs[0]), pointer(runs[1]))
        assert np.array_equal(runs[0], lowest)
    rng = np.random.default_rng(5)
    for _ in range(200):
        runs = [np.sort(rng.random(16)) for _ in range(2)]
        lowest = np.sort(np.concatenate(runs))[:16]
        library.lowest_of(pointer(runs[0]), pointer(runs[1]))
        assert np.array_equal(runs[0], lowest)


@pytest.mark.parametrize("stray", [np.float32(np.inf), np.float32(1e30), np.float32(1e-38), np.float32(np.nan), np.float32(0.0)])
@pytest.mark.parametrize("advance", [0, 1])
def test_a_walk_ends_by_the_windows_entries_alone(library, advance, stray):
    """Twelve rows hold distances 1, 2, ..; the three behind them, words of other lanes, hold ``stray``."""
    library.walk.argtypes = [C.c_void_p, C.c_int, C.c_void_p, C.c_int, C.c_float, C.c_float, C.c_int, C.c_void_p]
    for held in range(13):
        rows = np.full(15, stray, dtype=np.float32)
        rows[:held] = np.arange(1, held + 1)
        for first in range(held + 1):
            for passed in range(first, held + 1):        # entries before `first` are no farther than `passed`
                for limit in np.arange(first, held + 1.5, 0.5):
                    at, looked = np.array([first], dtype=np.int32), np.zeros(15, dtype=np.int32)
                    ended = library.walk(rows.ctypes.data, 15, at.ctypes.data, held, float(passed), float(limit), advance, looked.ctypes.data)
                    # what is left beyond a walk that ended is farther than the limit, and it ends wherever the window's last entry is
                    assert ended == (first < held and held > limit), (held, first, passed, limit)
                    assert np.all(looked <= 1) and not looked[held:].any() and not looked[:first].any()
                    assert looked[first:held].all() if not ended else looked[first:min(held, int(limit))].all()
                    assert first <= at[0] <= passed and (at[0] == first or advance)
                    if advance and not ended:
                        assert at[0] == passed


@pytest.mark.gpu
@pytest.mark.parametrize("sectors", [10, 14, 29, 41, 60, 80])
def test_lists_of_every_length_match_the_oracle(oracle, sectors):
    """Corridors seen end on: the longest lists have about as many entries as there are sectors, on 80 more than a column's own slots hold."""
    import launch_rules
    from random_cases import corridor_case
    from gradoom_amd import hostmath
    from gradoom_amd.renderer import HipRenderer, LaneState

    cameras = 6
    cosine = hostmath.cosine_correction("cpu").numpy()
    smap, tables, arrays = corridor_case(cameras, sectors)
    expected = torch.as_tensor(oracle.render(tables, arrays, cosine)["indexed"]).to("cuda:0")
    lanes = cameras                                         # no strip among the longest, whose columns share their lists
    while launch_rules.ask("select_strips", lanes, len(tables["walls"])) > 0:
        lanes += 32
    which = np.arange(lanes) % cameras
    renderer = HipRenderer(smap, lanes, "cuda:0", cosine_correction=cosine, tables=tables)
    indexed = torch.zeros((lanes, 240, 320), dtype=torch.uint8, device="cuda:0")
    renderer.render(LaneState.from_numpy({name: np.ascontiguousarray(value[which]) for name, value in arrays.items()}, "cuda:0"), indexed=indexed)
    torch.cuda.synchronize()
    assert renderer.status() == 0
    assert torch.equal(indexed, expected[torch.as_tensor(which, device="cuda:0")])
    renderer.close()
