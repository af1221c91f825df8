"""Billboard lists around the sizes at which the kernel changes its way (a chunk is 64 entries; a batch of 512 lanes and more
takes all rows of a strip at once), against the CPU oracle: byte for byte."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from random_cases import closed_door_parts  # noqa: E402

LANES = 4


@pytest.mark.parametrize("slots", [1, 63, 64, 65, 130, 512])
def test_billboard_lists_of_any_length_match_the_oracle(oracle, slots):
    from gradoom_amd import hostmath, mapbuild, synthmap
    from gradoom_amd.renderer import HipRenderer, LaneState
    from gradoom_amd.selfcheck import make_lane_arrays

    cosine = hostmath.cosine_correction("cpu").numpy()
    smap, poses, _sprites, _styles = closed_door_parts(301, LANES, variants=False)
    smap = synthmap.with_blend_tables(smap, 302)
    sprites = synthmap.generate_sprites(smap, LANES, slots, 303)
    rng = np.random.default_rng(slots)
    # every billboard before the eye, so that all of them are in the lists of the strips they reach; pairs at the same depth
    degrees = rng.uniform(-35, 35, (LANES, slots)) + poses.angle_bam[:, None].astype(np.float64) / 4294967296.0 * 360.0
    reach = rng.uniform(20, 400, (LANES, slots))
    sprites.x[...] = poses.x[:, None] + (reach * np.cos(np.deg2rad(degrees))).astype(np.float32)
    sprites.y[...] = poses.y[:, None] + (reach * np.sin(np.deg2rad(degrees))).astype(np.float32)
    sprites.x[:, 1::2], sprites.y[:, 1::2] = sprites.x[:, : slots - 1 : 2][:, : slots // 2], sprites.y[:, : slots - 1 : 2][:, : slots // 2]
    sprites.z[...] = poses.view_z[:, None] - 41.0 + rng.uniform(-30, 30, (LANES, slots)).astype(np.float32)
    arrays = make_lane_arrays(smap, poses, sprites)
    arrays["sprite_style"] = rng.choice(np.array([-1, -1, -2, 0, 1], dtype=np.int8), size=(LANES, slots))
    arrays["sprite_style"][::2] = -1                  # every other lane's billboards all plain
    tables = mapbuild.build_map_tables(smap)
    expected = torch.as_tensor(oracle.render(tables, arrays, cosine)["indexed"])
    for copies in (1, 128):                           # 4 lanes, 512 lanes
        lanes = LANES * copies
        tiled = {name: np.tile(value, (copies,) + (1,) * (value.ndim - 1)) for name, value in arrays.items()}
        renderer = HipRenderer(smap, lanes, "cuda:0", cosine_correction=cosine, tables=tables)
        indexed = torch.zeros((lanes, 240, 320), dtype=torch.uint8, device="cuda:0")
        renderer.render(LaneState.from_numpy(tiled, "cuda:0"), indexed=indexed)
        torch.cuda.synchronize()
        assert renderer.status() == 0
        assert torch.equal(indexed.cpu(), expected.repeat(copies, 1, 1)), lanes
        renderer.close()


@pytest.mark.parametrize("copies", [1, 128])   # quarters of a strip's rows, all rows at once
def test_eight_chunks_of_billboards_in_one_strip_match_the_oracle(oracle, copies):
    """All 512 slots a few degrees apart: one strip's list is painted in eight chunks, whose wavefronts end far apart since most
    billboards reach the last rows only."""

    from gradoom_amd import hostmath, mapbuild, synthmap
    from gradoom_amd.renderer import HipRenderer, LaneState
    from gradoom_amd.selfcheck import make_lane_arrays

    slots = 512
    cosine = hostmath.cosine_correction("cpu").numpy()
    smap, poses, _sprites, _styles = closed_door_parts(301, LANES, variants=False)
    smap = synthmap.with_blend_tables(smap, 302)
    sprites = synthmap.generate_sprites(smap, LANES, slots, 304)
    rng = np.random.default_rng(305)
    degrees = rng.uniform(2, 8, (LANES, slots)) + poses.angle_bam[:, None].astype(np.float64) / 4294967296.0 * 360.0
    reach = rng.uniform(20, 400, (LANES, slots))
    sprites.x[...] = poses.x[:, None] + (reach * np.cos(np.deg2rad(degrees))).astype(np.float32)
    sprites.y[...] = poses.y[:, None] + (reach * np.sin(np.deg2rad(degrees))).astype(np.float32)
    sprites.z[...] = poses.view_z[:, None] - 41.0 - (reach * rng.uniform(0, 0.4, (LANES, slots))).astype(np.float32)
    arrays = make_lane_arrays(smap, poses, sprites)
    arrays["sprite_style"] = rng.choice(np.array([-1, -1, -2, 0, 1], dtype=np.int8), size=(LANES, slots))
    arrays["sprite_style"][::2] = -1
    tables = mapbuild.build_map_tables(smap)
    expected = torch.as_tensor(oracle.render(tables, arrays, cosine)["indexed"])
    lanes = LANES * copies
    tiled = {name: np.tile(value, (copies,) + (1,) * (value.ndim - 1)) for name, value in arrays.items()}
    renderer = HipRenderer(smap, lanes, "cuda:0", cosine_correction=cosine, tables=tables)
    indexed = torch.zeros((lanes, 240, 320), dtype=torch.uint8, device="cuda:0")
    print(f"{lanes} lanes", flush=True)
    renderer.render(LaneState.from_numpy(tiled, "cuda:0"), indexed=indexed)
    torch.cuda.synchronize()
    assert renderer.status() == 0
    assert torch.equal(indexed.cpu(), expected.repeat(copies, 1, 1))
    renderer.close()


@pytest.mark.parametrize("slots", [6, 100])
@pytest.mark.parametrize("styles", [(0,), (-2, 1), (-1, 0, -2)])
def test_billboards_that_blend_over_the_flat_passes_pixels_match_the_oracle(oracle, slots, styles):
    """Cameras in the void look at billboards in front of the map: nothing is drawn below most of their pixels until the flat pass has been, which the
    early launch leaves to the late one; more of them than a chunk holds, and opaque ones among them."""

    from gradoom_amd import hostmath, mapbuild, synthmap
    from gradoom_amd.renderer import HipRenderer, LaneState
    from gradoom_amd.selfcheck import make_lane_arrays

    lanes = 6
    smap = synthmap.with_variant(synthmap.generate_map(81, grid=(6, 5), sectors=26, linedefs=180), 82, heights="uniform")
    smap = synthmap.with_blend_tables(smap, 83)
    poses = synthmap.generate_poses(smap, lanes, 84, margin=0.02)
    segments = np.asarray(smap.wall_segments, dtype=np.float64)
    rng = np.random.default_rng(85)
    poses.x[:4], poses.y[:4], poses.angle_bam[:4] = segments[:, [0, 2]].min() - 160, segments[:, [1, 3]].mean() + 40 * np.arange(4), 0
    sprites = synthmap.generate_sprites(smap, lanes, slots, 86)
    sprites.x[:4] = poses.x[:4, None] + rng.integers(30, 130, (4, slots))
    sprites.y[:4] = poses.y[:4, None] + rng.integers(-40, 41, (4, slots))
    sprites.z[:4] = poses.view_z[:4, None] - rng.integers(0, 60, (4, slots))
    arrays = make_lane_arrays(smap, poses, sprites)
    arrays["sprite_style"] = rng.choice(np.asarray(styles, dtype=np.int8), size=(lanes, slots))
    tables = mapbuild.build_map_tables(smap)
    cosine = hostmath.cosine_correction("cpu").numpy()
    expected = oracle.render(tables, arrays, cosine)["indexed"]
    opaque = oracle.render(tables, dict(arrays, sprite_style=np.full((lanes, slots), -1, dtype=np.int8)), cosine)["indexed"]
    assert (expected[:4] != opaque[:4]).sum() > 1000     # blending shows
    renderer = HipRenderer(smap, lanes, "cuda:0", cosine_correction=cosine, tables=tables)
    indexed = torch.zeros((lanes, 240, 320), dtype=torch.uint8, device="cuda:0")
    for _ in range(2):
        renderer.scribble(0xA5)
        renderer.render(LaneState.from_numpy(arrays, "cuda:0"), indexed=indexed)
        torch.cuda.synchronize()
        assert renderer.status() == 0
        assert np.array_equal(indexed.cpu().numpy(), expected)
    renderer.close()
