"""The layers over the walls (weapon, bullet chips) where their patches meet the edges of the view, against the CPU oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from random_cases import closed_door_case  # noqa: E402


@pytest.mark.parametrize("assembly", ["separate", "fused"])
def test_weapon_patches_at_and_past_every_edge_of_the_view_match_the_oracle(oracle, assembly):
    from gradoom_amd import hostmath, synthmap
    from gradoom_amd.renderer import HipRenderer, LaneState

    cosine = hostmath.cosine_correction("cpu").numpy()
    overlays = synthmap.generate_overlays(31)
    patches = len(overlays["weapon_w"])
    # each offset moves the patch from its place: off the left and the right edge, up and down, across each edge, beyond reach
    across = [0, -250, -180, 130, 190, 400, -(1 << 40), 1 << 40]
    down = [0, -150, -90, 60, 120, 300, -(1 << 40), 1 << 40]
    lanes = len(across) * len(down)
    smap, tables, arrays = closed_door_case(301, lanes)
    rng = np.random.default_rng(7)
    words = np.zeros((lanes, 5), dtype=np.int64)
    words[:, 0], words[:, 1] = rng.integers(0, patches, lanes), rng.integers(-1, patches, lanes)
    words[:, 2] = np.repeat(across, len(down)) * 65536 + rng.integers(0, 65536, lanes)
    words[:, 3] = np.tile(down, len(across)) * 65536 + rng.integers(0, 65536, lanes)
    words[:, 4] = 1
    arrays["weapon_state"] = words
    oracle.set_overlays(overlays)
    expected = oracle.render(tables, arrays, cosine)["indexed"]
    oracle.set_overlays(None)
    renderer = HipRenderer(smap, lanes, "cuda:0", cosine_correction=cosine, tables=tables)
    renderer.set_overlays(overlays)
    renderer.set_assembly(assembly)
    indexed = torch.zeros((lanes, 240, 320), dtype=torch.uint8, device="cuda:0")
    renderer.render(LaneState.from_numpy(arrays, "cuda:0"), indexed=indexed)
    torch.cuda.synchronize()
    assert renderer.status() == 0
    assert np.array_equal(indexed.cpu().numpy(), expected)
    renderer.close()


@pytest.mark.parametrize("where", ["inside", "outside"])
def test_chips_over_pixels_of_every_kind_match_the_oracle(oracle, where):
    """Chips cut off by tiers, planes and masked textures before them, and (cameras in the void) chips whose rows reach pixels that show
    the flat pass's picture, resolved, repaired and not."""
    import sys
    import types

    from conftest import ROOT
    from gradoom_amd import hostmath, mapbuild, overlay_inputs, synthmap
    from gradoom_amd.renderer import HipRenderer, LaneState
    from gradoom_amd.selfcheck import make_lane_arrays
    from random_cases import closed_door_parts, outside_parts

    sys.path.insert(0, f"{ROOT}/tests/golden")
    import refdrive

    cosine = hostmath.cosine_correction("cpu").numpy()
    overlays = synthmap.generate_overlays(32)
    lanes, slots = 16, 64
    smap, poses, sprites = closed_door_parts(305, lanes, mixed=True)[:3] if where == "inside" else outside_parts(lanes)
    tables = mapbuild.build_map_tables(smap)
    arrays = make_lane_arrays(smap, poses, sprites)
    engine = types.SimpleNamespace(num_envs=lanes, hitscan_decal_slots=slots, **{name: arrays[name] for name in ("x", "y", "angle", "view_z")})
    for name, dtype, value in (("wall", torch.int64, 0), ("along", torch.float32, 0), ("z", torch.float32, 0), ("style", torch.int64, 0), ("serial", torch.int64, -1)):
        setattr(engine, "hitscan_decal_" + name, torch.full((lanes, slots), value, dtype=dtype))
    refdrive.set_decals(engine, smap, 306)
    state, geometry = overlay_inputs.decal_inputs(
        engine.hitscan_decal_serial, engine.hitscan_decal_wall, engine.hitscan_decal_along, engine.hitscan_decal_z, engine.hitscan_decal_style,
        torch.as_tensor(np.asarray(tables["walls"], dtype=np.float32)), overlay_inputs.fine_sine_fixed(),
    )
    plain = oracle.render(tables, arrays, cosine)["indexed"]
    arrays["decal_state"], arrays["decal_geom"] = state.numpy(), geometry.numpy()
    oracle.set_overlays(overlays)
    expected = oracle.render(tables, arrays, cosine)["indexed"]
    oracle.set_overlays(None)
    assert (expected != plain).any()                  # some chips show
    renderer = HipRenderer(smap, lanes, "cuda:0", cosine_correction=cosine, tables=tables)
    renderer.set_overlays(overlays)
    renderer.scribble(0xFF)
    indexed = torch.zeros((lanes, 240, 320), dtype=torch.uint8, device="cuda:0")
    renderer.render(LaneState.from_numpy(arrays, "cuda:0"), indexed=indexed)
    torch.cuda.synchronize()
    assert renderer.status() == 0
    assert np.array_equal(indexed.cpu().numpy(), expected)
    renderer.close()


@pytest.mark.parametrize("assembly", ["separate", "fused"])
@pytest.mark.parametrize("patches", [None, 40, 1])
def test_status_bars_of_every_kind_of_number_match_the_oracle(oracle, assembly, patches):
    """Numbers of one to three digits and beyond, with and without a sign, faces that are no patches, offsets that move glyphs past the bar's edges,
    and lists whose last patches do not exist."""
    from gradoom_amd import hostmath, synthmap
    from gradoom_amd.renderer import HipRenderer, LaneState

    cosine = hostmath.cosine_correction("cpu").numpy()
    overlays = dict(synthmap.generate_overlays(33))
    rng = np.random.default_rng(11)
    for name, reach in (("hud_left", 12), ("hud_top", 20)):
        overlays[name] = (overlays[name] + rng.integers(-reach, reach + 1, overlays[name].shape)).astype(overlays[name].dtype)
    count = patches or len(overlays["hud_w"])
    whole = dict(overlays, hud_w=overlays["hud_w"].copy())
    whole["hud_w"][count:] = 0                       # what the oracle is given for the patches that the renderer's list ends before
    overlays.update({name: overlays[name][:count] for name in overlays if name.startswith("hud_")})
    numbers = np.array([0, 1, 9, 10, 99, 100, 999, 1000, -1, -9, -10, -99, -100, 2**31 - 1, -(2**31), 50, 300], dtype=np.int64)
    lanes = 48
    smap, tables, arrays = closed_door_case(301, lanes)
    words = numbers[rng.integers(0, len(numbers), (lanes, 9))]
    words[:, 3] = rng.integers(-2, count + 3, lanes)
    words[:, 4] = rng.integers(0, 64, lanes)
    arrays["hud_state"] = words.astype(np.int32)
    oracle.set_overlays(whole)
    expected = oracle.render(tables, arrays, cosine)["indexed"]
    oracle.set_overlays(None)
    assert len({bar.tobytes() for bar in expected[:, 208:]}) > (0 if patches == 1 else 20)
    renderer = HipRenderer(smap, lanes, "cuda:0", cosine_correction=cosine, tables=tables)
    renderer.set_overlays(overlays)
    renderer.set_assembly(assembly)
    indexed = torch.zeros((lanes, 240, 320), dtype=torch.uint8, device="cuda:0")
    renderer.render(LaneState.from_numpy(arrays, "cuda:0"), indexed=indexed)
    torch.cuda.synchronize()
    assert np.array_equal(indexed.cpu().numpy(), expected)
    renderer.close()


@pytest.mark.parametrize("slots, chips", [(3, 1), (63, 40), (64, 40), (65, 40), (200, 130)])
def test_chips_in_any_number_of_slots_match_the_oracle(oracle, slots, chips):
    """A chunk of decal_kernel is 64 slots; the chips of several chunks are painted in the order of their slots all the same."""
    import sys
    import types

    from conftest import ROOT
    from gradoom_amd import hostmath, overlay_inputs, synthmap
    from gradoom_amd.renderer import HipRenderer, LaneState

    sys.path.insert(0, f"{ROOT}/tests/golden")
    import refdrive

    cosine = hostmath.cosine_correction("cpu").numpy()
    overlays = synthmap.generate_overlays(34)
    lanes = 4
    smap, tables, arrays = closed_door_case(303, lanes)
    engine = types.SimpleNamespace(num_envs=lanes, hitscan_decal_slots=slots, **{name: arrays[name] for name in ("x", "y", "angle", "view_z")})
    for name, dtype, value in (("wall", torch.int64, 0), ("along", torch.float32, 0), ("z", torch.float32, 0), ("style", torch.int64, 0), ("serial", torch.int64, -1)):
        setattr(engine, "hitscan_decal_" + name, torch.full((lanes, slots), value, dtype=dtype))
    refdrive.set_decals(engine, smap, 35, per_lane=chips)
    state, geometry = overlay_inputs.decal_inputs(
        engine.hitscan_decal_serial, engine.hitscan_decal_wall, engine.hitscan_decal_along, engine.hitscan_decal_z, engine.hitscan_decal_style,
        torch.as_tensor(np.asarray(tables["walls"], dtype=np.float32)), overlay_inputs.fine_sine_fixed(),
    )
    bare = oracle.render(tables, arrays, cosine)["indexed"]
    arrays["decal_state"], arrays["decal_geom"] = state.numpy(), geometry.numpy()
    oracle.set_overlays(overlays)
    expected = oracle.render(tables, arrays, cosine)["indexed"]
    oracle.set_overlays(None)
    assert chips == 1 or (expected != bare).any()
    renderer = HipRenderer(smap, lanes, "cuda:0", cosine_correction=cosine, tables=tables)
    renderer.set_overlays(overlays)
    indexed = torch.zeros((lanes, 240, 320), dtype=torch.uint8, device="cuda:0")
    renderer.render(LaneState.from_numpy(arrays, "cuda:0"), indexed=indexed)
    torch.cuda.synchronize()
    assert renderer.status() == 0
    assert np.array_equal(indexed.cpu().numpy(), expected)
    renderer.close()
