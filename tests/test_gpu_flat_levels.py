"""The flat pass at the sizes where its probes change path: too few plane levels for the bit sets, one bit-set word and a few,
more levels named by a bucket than a pixel's or a row's list holds, more levels than the bit sets cover."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sectors", [20, 33, 40, 150, 520])
def test_flat_pass_with_a_plane_level_per_sector_matches_the_oracle(oracle, sectors):
    from gradoom_amd import hostmath, mapbuild, synthmap
    from gradoom_amd.renderer import HipRenderer, LaneState
    from gradoom_amd.selfcheck import make_lane_arrays

    lanes = 4
    side = int(np.ceil(np.sqrt(sectors * 1.15)))
    smap = synthmap.with_variant(synthmap.generate_map(60 + sectors, grid=(side, side), sectors=sectors, linedefs=7 * sectors), 61, heights="uniform")
    poses = synthmap.generate_poses(smap, lanes, 62, pitch=True, margin=0.02)
    # half of the cameras in the void beside the map, looking at it: most of their screens is the flat pass's
    segments = np.asarray(smap.wall_segments, dtype=np.float64)
    poses.x[1], poses.y[1], poses.angle_bam[1] = segments[:, [0, 2]].min() - 60, segments[:, [1, 3]].mean(), 0
    poses.x[3], poses.y[3], poses.angle_bam[3] = segments[:, [0, 2]].mean(), segments[:, [1, 3]].max() + 25, 3 << 30
    arrays = make_lane_arrays(smap, poses, synthmap.generate_sprites(smap, lanes, 8, 63))
    tables = mapbuild.build_map_tables(smap)
    cosine = hostmath.cosine_correction("cpu").numpy()
    expected = oracle.render(tables, arrays, cosine)
    renderer = HipRenderer(smap, lanes, "cuda:0", cosine_correction=cosine, tables=tables)
    indexed = torch.zeros((lanes, 240, 320), dtype=torch.uint8, device="cuda:0")
    print(f"{sectors} sectors, {len(tables['floor_levels'])} + {len(tables['ceil_levels'])} levels", flush=True)
    renderer.render(LaneState.from_numpy(arrays, "cuda:0"), indexed=indexed)
    torch.cuda.synchronize()
    assert renderer.status() == 0
    assert np.array_equal(indexed.cpu().numpy(), expected["indexed"])
    renderer.close()


@pytest.mark.parametrize("degrees", [0, 12, 30])
def test_repairs_of_tall_screen_halves_match_the_oracle(oracle, degrees):
    """Cameras in the void look at the map, level and up or down: the rows to repair reach over a half of the screen of 104 rows, of
    more than the 108 that flat_span_finish_kernel holds at a time, and of nearly all 208."""
    from gradoom_amd import hostmath, mapbuild, synthmap
    from gradoom_amd.renderer import HipRenderer, LaneState
    from gradoom_amd.selfcheck import make_lane_arrays

    lanes = 4
    smap = synthmap.with_variant(synthmap.generate_map(71, grid=(7, 6), sectors=36, linedefs=250), 72, heights="uniform")
    poses = synthmap.generate_poses(smap, lanes, 73, margin=0.02)
    segments = np.asarray(smap.wall_segments, dtype=np.float64)
    for lane, sign in enumerate((1, -1, 1, -1)):
        if lane < 2:
            poses.x[lane], poses.y[lane], poses.angle_bam[lane] = segments[:, [0, 2]].min() - 60, segments[:, [1, 3]].mean(), 0
        else:
            poses.x[lane], poses.y[lane], poses.angle_bam[lane] = segments[:, [0, 2]].mean(), segments[:, [1, 3]].max() + 25, 3 << 30
        poses.pitch_bam[lane] = sign * degrees * (182 << 16)
    arrays = make_lane_arrays(smap, poses, synthmap.generate_sprites(smap, lanes, 8, 74))
    tables = mapbuild.build_map_tables(smap)
    cosine = hostmath.cosine_correction("cpu").numpy()
    expected = oracle.render(tables, arrays, cosine)
    renderer = HipRenderer(smap, lanes, "cuda:0", cosine_correction=cosine, tables=tables)
    indexed = torch.zeros((lanes, 240, 320), dtype=torch.uint8, device="cuda:0")
    renderer.scribble(0xA5)
    renderer.render(LaneState.from_numpy(arrays, "cuda:0"), indexed=indexed)
    torch.cuda.synchronize()
    assert renderer.status() == 0
    assert np.array_equal(indexed.cpu().numpy(), expected["indexed"])
    renderer.close()
