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
    words[:, 0], words[:, 1] = rng.integers(-1, patches + 1, lanes), rng.integers(-1, patches + 1, lanes)   # none, and one past the last
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
