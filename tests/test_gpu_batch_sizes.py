"""Batches of many sizes, and on either side of those at which the traversal shares a strip out over more or fewer wavefronts: every
lane's frame is the one the CPU oracle draws for its camera."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from random_cases import closed_door_parts  # noqa: E402

CAMERAS = 5


@pytest.mark.parametrize("lanes", [1, 5, 25, 26, 103, 640, 641, 1535, 1536])
def test_batches_around_the_sizes_of_the_traversals_rules_match_the_oracle(oracle, lanes):
    from gradoom_amd import hostmath, mapbuild
    from gradoom_amd.renderer import HipRenderer, LaneState
    from gradoom_amd.selfcheck import make_lane_arrays

    cosine = hostmath.cosine_correction("cpu").numpy()
    smap, poses, sprites, styles = closed_door_parts(6002, CAMERAS, mixed=True)
    arrays = make_lane_arrays(smap, poses, sprites)
    arrays["sprite_style"] = styles
    tables = mapbuild.build_map_tables(smap)
    expected = torch.as_tensor(oracle.render(tables, arrays, cosine)["indexed"]).to("cuda:0")
    which = np.arange(lanes) % CAMERAS
    renderer = HipRenderer(smap, lanes, "cuda:0", cosine_correction=cosine, tables=tables)
    indexed = torch.zeros((lanes, 240, 320), dtype=torch.uint8, device="cuda:0")
    state = LaneState.from_numpy({name: np.ascontiguousarray(value[which]) for name, value in arrays.items()}, "cuda:0")
    renderer.render(state, indexed=indexed)
    torch.cuda.synchronize()
    assert renderer.status() == 0
    assert torch.equal(indexed, expected[torch.as_tensor(which, device="cuda:0")])
    renderer.close()


@pytest.mark.parametrize("rule", ["selection", "four_parts", "two_parts"])
def test_batches_on_both_sides_of_a_sharing_rules_line_match_the_oracle(oracle, rule):
    """Lines that sharing rules have had, the first of them following the map's linedefs.  (Where they lie now: test_gpu_shared_columns.py and
    test_gpu_shared_lists.py.)"""

    from gradoom_amd import hostmath, mapbuild
    from gradoom_amd.renderer import HipRenderer, LaneState
    from gradoom_amd.selfcheck import make_lane_arrays

    cosine = hostmath.cosine_correction("cpu").numpy()
    smap, poses, sprites, styles = closed_door_parts(6002, CAMERAS, mixed=True)
    arrays = make_lane_arrays(smap, poses, sprites)
    arrays["sprite_style"] = styles
    tables = mapbuild.build_map_tables(smap)
    expected = torch.as_tensor(oracle.render(tables, arrays, cosine)["indexed"]).to("cuda:0")
    linedefs = len(tables["walls"])
    assert linedefs < 4096
    line = {"selection": 192 + linedefs // 4, "four_parts": 561, "two_parts": 1345}[rule]
    renderer = HipRenderer(smap, line, "cuda:0", cosine_correction=cosine, tables=tables)
    for lanes in (line - 1, line):
        print(f"{rule}: {lanes} lanes", flush=True)
        which = np.arange(lanes) % CAMERAS
        indexed = torch.zeros((lanes, 240, 320), dtype=torch.uint8, device="cuda:0")
        state = LaneState.from_numpy({name: np.ascontiguousarray(value[which]) for name, value in arrays.items()}, "cuda:0")
        renderer.render(state, indexed=indexed)
        torch.cuda.synchronize()
        assert renderer.status() == 0
        assert torch.equal(indexed, expected[torch.as_tensor(which, device="cuda:0")])
    renderer.close()
