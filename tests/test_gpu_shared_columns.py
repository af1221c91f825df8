"""Columns that share a wavefront's lanes: on either side of the batch sizes at which a column has sixteen lanes, eight, four, two or one, every
lane's frame is the one the CPU oracle draws for its camera, wall depths (which chips are drawn against) among it."""

from __future__ import annotations

import sys
import types

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

CAMERAS, SLOTS = 16, 64


@pytest.mark.parametrize("chips", [False, True])
@pytest.mark.parametrize("inverted", [False, True])
def test_batches_at_the_lines_of_the_columns_shares_match_the_oracle(oracle, inverted, chips):
    import launch_rules
    from conftest import ROOT
    from gradoom_amd import hostmath, mapbuild, overlay_inputs, synthmap
    from gradoom_amd.renderer import HipRenderer, LaneState
    from gradoom_amd.selfcheck import make_lane_arrays
    from random_cases import closed_door_parts

    sys.path.insert(0, f"{ROOT}/tests/golden")
    import refdrive

    cosine = hostmath.cosine_correction("cpu").numpy()
    overlays = synthmap.generate_overlays(32) if chips else None
    smap, poses, sprites, styles = closed_door_parts(411 + inverted, CAMERAS, mixed=True, inverted=inverted, eye_any=True)
    tables = mapbuild.build_map_tables(smap)
    arrays = make_lane_arrays(smap, poses, sprites)
    arrays["sprite_style"] = styles
    if chips:
        engine = types.SimpleNamespace(num_envs=CAMERAS, hitscan_decal_slots=SLOTS, **{name: arrays[name] for name in ("x", "y", "angle", "view_z")})
        for name, dtype, value in (("wall", torch.int64, 0), ("along", torch.float32, 0), ("z", torch.float32, 0), ("style", torch.int64, 0), ("serial", torch.int64, -1)):
            setattr(engine, "hitscan_decal_" + name, torch.full((CAMERAS, SLOTS), value, dtype=dtype))
        refdrive.set_decals(engine, smap, 412)
        state, geometry = overlay_inputs.decal_inputs(
            engine.hitscan_decal_serial, engine.hitscan_decal_wall, engine.hitscan_decal_along, engine.hitscan_decal_z, engine.hitscan_decal_style,
            torch.as_tensor(np.asarray(tables["walls"], dtype=np.float32)), overlay_inputs.fine_sine_fixed(),
        )
        arrays["decal_state"], arrays["decal_geom"] = state.numpy(), geometry.numpy()
    oracle.set_overlays(overlays)
    expected = torch.as_tensor(oracle.render(tables, arrays, cosine)["indexed"]).to("cuda:0")
    oracle.set_overlays(None)
    lines = launch_rules.lines("raster_sixteen") + launch_rules.lines("raster_parts")
    assert len(lines) == 4 and lines == sorted(lines)      # sixteen lanes a column go before what raster_parts says
    for lanes in sorted({1} | set(lines) | {line - 1 for line in lines}):
        print(f"{lanes} lanes", flush=True)
        which = np.arange(lanes) % CAMERAS
        renderer = HipRenderer(smap, lanes, "cuda:0", cosine_correction=cosine, tables=tables)
        if overlays is not None:
            renderer.set_overlays(overlays)
        renderer.scribble(0xA5)
        indexed = torch.zeros((lanes, 240, 320), dtype=torch.uint8, device="cuda:0")
        renderer.render(LaneState.from_numpy({name: np.ascontiguousarray(value[which]) for name, value in arrays.items()}, "cuda:0"), indexed=indexed)
        torch.cuda.synchronize()
        assert renderer.status() == 0
        assert torch.equal(indexed, expected[torch.as_tensor(which, device="cuda:0")])
        renderer.close()
