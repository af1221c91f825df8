"""The tables that a work-group of the walls' drawing keeps in LDS (texture sizes, which of them are no powers of two, 224 textures at most) at the
edges of their words and where they no longer hold all textures, against the CPU oracle."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

LANES = 4


@pytest.mark.parametrize("textures", [31, 32, 33, 64, 65, 193, 223, 224, 225, 260])
def test_any_number_of_textures_matches_the_oracle(oracle, textures):
    from gradoom_amd import hostmath, mapbuild, synthmap
    from gradoom_amd.renderer import HipRenderer, LaneState
    from gradoom_amd.selfcheck import make_lane_arrays

    cosine = hostmath.cosine_correction("cpu").numpy()
    smap = synthmap.generate_map(515, grid=(7, 6), sectors=36, linedefs=260, midtex=0.2, wall_textures=textures - 12, flats=12)
    smap = synthmap.with_variant(smap, 516, heights="uniform", textures="npot")
    assert len(smap.texture_widths) == textures
    poses = synthmap.generate_poses(smap, LANES, 517, pitch=True, margin=0.02)
    arrays = make_lane_arrays(smap, poses, synthmap.generate_sprites(smap, LANES, 8, 518))
    tables = mapbuild.build_map_tables(smap)
    expected = torch.as_tensor(oracle.render(tables, arrays, cosine)["indexed"])
    renderer = HipRenderer(smap, LANES, "cuda:0", cosine_correction=cosine, tables=tables)
    lanes = LaneState.from_numpy(arrays, "cuda:0")
    for assembly in ("auto", "fused"):
        renderer.set_assembly(assembly)
        renderer.scribble(0x5A)
        indexed = torch.zeros((LANES, 240, 320), dtype=torch.uint8, device="cuda:0")
        renderer.render(lanes, indexed=indexed)
        torch.cuda.synchronize()
        assert renderer.status() == 0
        assert torch.equal(indexed.cpu(), expected), assembly
    renderer.close()
