"""Batches of many sizes, and on either side of those at which a rule on batch sizes changes how a frame's launches are cut: every lane's
frame is the one the CPU oracle draws for its camera."""

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
    """Lines that sharing rules once had, kept as more batch sizes.  (Those of today's rules: below, and in test_gpu_shared_columns.py and
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


# (those of the selection and of the drawing: test_gpu_shared_lists.py and test_gpu_shared_columns.py)
@pytest.mark.parametrize("rule, billboards", [
    ("setup_whole_lanes", True), ("select_together", True), ("raster_sixteen", True), ("geometry_parts", True), ("gap_waves", True), ("sprite_row_parts", True), ("side_stream_pays", True), ("side_stream_pays", False),
])
def test_batches_on_both_sides_of_a_rules_line_match_the_oracle(oracle, rule, billboards):
    import launch_rules
    from gradoom_amd import hostmath, mapbuild, synthmap
    from gradoom_amd.renderer import HipRenderer, LaneState
    from gradoom_amd.selfcheck import make_lane_arrays

    cosine = hostmath.cosine_correction("cpu").numpy()
    smap = synthmap.generate_map(6003, grid=(9, 9), sectors=64, linedefs=600, layout="brick", midtex=0.1)      # too many linedefs for a work-group
    smap = synthmap.with_variant(smap, 6004, heights="doors", textures="npot", lights=True)
    poses = synthmap.generate_poses(smap, CAMERAS, 6005, pitch=True, flash=True, margin=0.005)
    arrays = make_lane_arrays(smap, poses, synthmap.generate_sprites(smap, CAMERAS, 16 if billboards else 0, 6006))
    tables = mapbuild.build_map_tables(smap)
    expected = torch.as_tensor(oracle.render(tables, arrays, cosine)["indexed"]).to("cuda:0")
    other = {launch_rules.LINEDEFS: len(tables["walls"]), launch_rules.BILLBOARDS: billboards, launch_rules.NOTHING: 0}[launch_rules.RULES[rule]]
    lines = launch_rules.lines(rule, other)
    assert lines
    for lanes in sorted(set(lines) | {line - 1 for line in lines}):
        print(f"{rule}: {lanes} lanes", flush=True)
        which = np.arange(lanes) % CAMERAS
        renderer = HipRenderer(smap, lanes, "cuda:0", cosine_correction=cosine, tables=tables)
        indexed = torch.zeros((lanes, 240, 320), dtype=torch.uint8, device="cuda:0")
        state = LaneState.from_numpy({name: np.ascontiguousarray(value[which]) for name, value in arrays.items()}, "cuda:0")
        renderer.render(state, indexed=indexed)
        torch.cuda.synchronize()
        assert renderer.status() == 0
        assert torch.equal(indexed, expected[torch.as_tensor(which, device="cuda:0")])
        renderer.close()


def test_batches_at_the_lines_of_large_maps_gap_columns_match_the_oracle(oracle):
    """Maps of 3000 linedefs and more have lines of their own; a plane level per sector, and cameras off the map, whose frames are mostly gap pixels."""
    import launch_rules
    from gradoom_amd import hostmath, mapbuild, synthmap
    from gradoom_amd.renderer import HipRenderer, LaneState
    from gradoom_amd.selfcheck import make_lane_arrays

    cosine = hostmath.cosine_correction("cpu").numpy()
    smap = synthmap.with_variant(synthmap.generate_map(6007, grid=(19, 18), sectors=310, linedefs=3050, midtex=0.1), 6008, heights="uniform")
    poses = synthmap.generate_poses(smap, CAMERAS, 6009, pitch=True, margin=0.02)
    segments = np.asarray(smap.wall_segments, dtype=np.float64)
    for camera in (1, 3):
        poses.x[camera], poses.y[camera], poses.angle_bam[camera] = segments[:, [0, 2]].min() - 60 * camera, segments[:, [1, 3]].mean(), 0
    arrays = make_lane_arrays(smap, poses, synthmap.generate_sprites(smap, CAMERAS, 32, 6010))
    tables = mapbuild.build_map_tables(smap)
    linedefs = len(tables["walls"])
    lines = launch_rules.lines("gap_waves", linedefs)
    assert linedefs >= 3000 and lines != launch_rules.lines("gap_waves", 600) and len(lines) == 2
    expected = torch.as_tensor(oracle.render(tables, arrays, cosine)["indexed"]).to("cuda:0")
    for lanes in sorted(set(lines) | {line - 1 for line in lines}):
        print(f"{lanes} lanes", flush=True)
        which = np.arange(lanes) % CAMERAS
        renderer = HipRenderer(smap, lanes, "cuda:0", cosine_correction=cosine, tables=tables)
        indexed = torch.zeros((lanes, 240, 320), dtype=torch.uint8, device="cuda:0")
        renderer.render(LaneState.from_numpy({name: np.ascontiguousarray(value[which]) for name, value in arrays.items()}, "cuda:0"), indexed=indexed)
        torch.cuda.synchronize()
        assert renderer.status() == 0
        assert torch.equal(indexed, expected[torch.as_tensor(which, device="cuda:0")])
        renderer.close()
