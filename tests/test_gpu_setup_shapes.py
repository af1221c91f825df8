"""Linedef setup on either side of its rules: a work-group for a whole lane or one for 256 linedefs (up to 512 linedefs, from 800
lanes), and lanes with more linedefs than are sorted at a time (4096), against the CPU oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

LANES = 4


@pytest.mark.parametrize("linedefs, lanes", [(512, 4), (513, 4), (513, 796), (513, 800), (4224, 4), (4224, 800)])
def test_linedef_setup_of_every_shape_matches_the_oracle(oracle, linedefs, lanes):
    from gradoom_amd import hostmath, mapbuild, synthmap
    from gradoom_amd.renderer import HipRenderer, LaneState
    from gradoom_amd.selfcheck import make_lane_arrays

    cosine = hostmath.cosine_correction("cpu").numpy()
    grid, sectors = ((8, 8), 58) if linedefs < 1000 else ((21, 21), 400)
    smap = synthmap.generate_map(411, grid=grid, sectors=sectors, linedefs=linedefs, midtex=0.2)
    assert len(smap.wall_segments) == linedefs
    poses = synthmap.generate_poses(smap, LANES, 412, pitch=True, margin=0.02)
    arrays = make_lane_arrays(smap, poses, synthmap.generate_sprites(smap, LANES, 8, 413))
    tables = mapbuild.build_map_tables(smap)
    expected = torch.as_tensor(oracle.render(tables, arrays, cosine)["indexed"])
    copies = lanes // LANES
    tiled = {name: np.tile(value, (copies,) + (1,) * (value.ndim - 1)) for name, value in arrays.items()}
    renderer = HipRenderer(smap, lanes, "cuda:0", cosine_correction=cosine, tables=tables)
    renderer.scribble(0x5A)
    indexed = torch.zeros((lanes, 240, 320), dtype=torch.uint8, device="cuda:0")
    renderer.render(LaneState.from_numpy(tiled, "cuda:0"), indexed=indexed)
    torch.cuda.synchronize()
    assert renderer.status() == 0
    assert torch.equal(indexed.cpu(), expected.repeat(copies, 1, 1))
    renderer.close()
