"""The selection's columns that share their candidate lists out over 8, 16 or 32 lanes: on either side of the lines at which their number
changes, and with all of a batch's strips, some of them or none among the longest, every lane's frame is the one the CPU oracle draws."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

CAMERAS = 4


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("linedefs", [320, 700, 1100])
def test_batches_at_the_lines_of_the_lists_shares_match_the_oracle(oracle, linedefs, split):
    import launch_rules
    from gradoom_amd import hostmath, mapbuild, synthmap
    from gradoom_amd.renderer import HipRenderer, LaneState
    from gradoom_amd.selfcheck import make_lane_arrays

    cosine = hostmath.cosine_correction("cpu").numpy()
    cells = {320: 7, 700: 10, 1100: 12}[linedefs]
    smap = synthmap.generate_map(linedefs, grid=(cells, cells), sectors=cells * cells * 4 // 5, linedefs=linedefs, layout="brick", midtex=0.1)
    smap = synthmap.with_variant(smap, linedefs + 1, heights="doors", textures="npot", lights=True)
    if split:
        smap = synthmap.split_linedefs(smap, linedefs + 2)
    poses = synthmap.generate_poses(smap, CAMERAS, linedefs + 3, pitch=True, flash=True, margin=0.005)
    arrays = make_lane_arrays(smap, poses, synthmap.generate_sprites(smap, CAMERAS, 16, linedefs + 4))
    tables = mapbuild.build_map_tables(smap)
    expected = torch.as_tensor(oracle.render(tables, arrays, cosine)["indexed"]).to("cuda:0")
    count = len(tables["walls"])
    assert count >= linedefs
    lines = {launch_rules.ask("select_strips", 1, count) // 5 + 1}                   # the first batch beyond each: some strips are not among the longest
    lines.update(launch_rules.lines("select_strips", count), launch_rules.lines("select_lanes", count))
    for lanes in sorted({1} | lines | {line - 1 for line in lines}):
        print(f"{count} linedefs: {lanes} lanes", flush=True)
        which = np.arange(lanes) % CAMERAS
        renderer = HipRenderer(smap, lanes, "cuda:0", cosine_correction=cosine, tables=tables)
        indexed = torch.zeros((lanes, 240, 320), dtype=torch.uint8, device="cuda:0")
        renderer.render(LaneState.from_numpy({name: np.ascontiguousarray(value[which]) for name, value in arrays.items()}, "cuda:0"), indexed=indexed)
        torch.cuda.synchronize()
        assert renderer.status() == 0
        assert torch.equal(indexed, expected[torch.as_tensor(which, device="cuda:0")])
        renderer.close()


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("linedefs", [1720, 2350, 3050])
def test_large_maps_at_the_lines_of_the_selections_rules_match_the_oracle(oracle, linedefs, split):
    """Beyond the line of select_together the longest strips and the others are two launches on two streams: on maps of these sizes some strips are
    among the longest there, and not all are."""
    import launch_rules
    from gradoom_amd import hostmath, mapbuild, synthmap
    from gradoom_amd.renderer import HipRenderer, LaneState
    from gradoom_amd.selfcheck import make_lane_arrays

    cosine = hostmath.cosine_correction("cpu").numpy()
    cells = {1720: 15, 2350: 17, 3050: 20}[linedefs]
    smap = synthmap.generate_map(linedefs, grid=(cells, cells), sectors=cells * cells * 4 // 5, linedefs=linedefs, midtex=0.1)
    smap = synthmap.with_variant(smap, linedefs + 1, heights="doors", textures="npot", lights=True)
    if split:
        smap = synthmap.split_linedefs(smap, linedefs + 2)
    poses = synthmap.generate_poses(smap, CAMERAS, linedefs + 3, pitch=True, flash=True, margin=0.005)
    arrays = make_lane_arrays(smap, poses)
    tables = mapbuild.build_map_tables(smap)
    count = len(tables["walls"])
    together = launch_rules.lines("select_together")
    assert len(together) == 1 and launch_rules.ask("select_together", together[0]) == 0
    for lanes in (together[0] - 1, together[0]):
        assert 0 < launch_rules.ask("select_strips", lanes, count) < 5 * lanes
    expected = torch.as_tensor(oracle.render(tables, arrays, cosine)["indexed"]).to("cuda:0")
    lines = {*together, *launch_rules.lines("select_strips", count), *launch_rules.lines("select_lanes", count)}
    lines.update(launch_rules.ask("select_strips", lanes, count) // 5 + 1 for lanes in (1, min(lines)))     # the first batches of which some strips are not among the longest
    renderer = HipRenderer(smap, max(lines), "cuda:0", cosine_correction=cosine, tables=tables)
    for lanes in sorted(lines | {line - 1 for line in lines}):
        print(f"{count} linedefs: {lanes} lanes", flush=True)
        which = np.arange(lanes) % CAMERAS
        indexed = torch.zeros((lanes, 240, 320), dtype=torch.uint8, device="cuda:0")
        renderer.render(LaneState.from_numpy({name: np.ascontiguousarray(value[which]) for name, value in arrays.items()}, "cuda:0"), indexed=indexed)
        torch.cuda.synchronize()
        assert renderer.status() == 0
        assert torch.equal(indexed, expected[torch.as_tensor(which, device="cuda:0")])
    renderer.close()
