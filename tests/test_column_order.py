"""The sorting networks that order the nearest entries of a column's list (``csrc/gd_order.h``), compiled for the host; and columns with lists of one to six
such windows, drawn with a lane a column, against the CPU oracle."""

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
"""


def test_the_networks_order_numbers(tmp_path):
    path = str(tmp_path / "liborder.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-Wno-unknown-pragmas", "-I", CSRC, "-x", "c++", "-o", path, "-"], input=DRIVER, text=True, check=True)
    library = C.CDLL(path)
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
