"""The sorting network that orders a column's list (``csrc/gd_order.h``), compiled for the host; and columns with lists of every length that the selection
orders by a network of its own, drawn with a lane a column, against the CPU oracle."""

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
template <int COUNT> static void order(unsigned *v) {
    unsigned (&w)[COUNT] = *reinterpret_cast<unsigned (*)[COUNT]>(v);
    order_up(w);
}
extern "C" void order_numbers(unsigned *v, int count) {
    switch (count) { case 32: order<32>(v); break; case 48: order<48>(v); break; case 64: order<64>(v); break; }
}
"""


@pytest.mark.parametrize("count", [32, 48, 64])
def test_the_network_orders_numbers(tmp_path, count):
    path = str(tmp_path / "liborder.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-Wno-unknown-pragmas", "-I", CSRC, "-x", "c++", "-o", path, "-"], input=DRIVER, text=True, check=True)
    order = C.CDLL(path).order_numbers
    rng = np.random.default_rng(count)
    for share in np.linspace(0.0, 1.0, count + 1):          # zeros and ones (what a network orders of these it orders of all numbers), then any numbers
        for numbers in (rng.random((40, count)) < share).astype(np.uint32), rng.integers(0, 1 << 32, (40, count), dtype=np.uint32):
            for row in numbers:
                ordered = row.copy()
                order(ordered.ctypes.data_as(C.c_void_p), count)
                assert np.array_equal(ordered, np.sort(row))


@pytest.mark.gpu
@pytest.mark.parametrize("sectors", [10, 29, 41, 46, 60, 80])
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
