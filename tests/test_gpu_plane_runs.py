"""Plane shading where a tile of the view (64 columns, 16 rows) holds more runs of pixels than a wavefront works out at once, and (the
smaller cells) lanes that draw two thousand linedefs, more than the wavefronts of wall_geometry_kernel list at once, against the CPU
oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

LANES = 6


def _runs(depth):
    """At least as many runs as this begin in the most varied tile: stretches of three or more columns of a row at one depth."""
    most = 0
    for y in range(0, 208, 16):
        for x in range(0, 320, 64):
            runs = 0
            for row in depth[y : y + 16, x : x + 64]:
                cuts = np.concatenate([[0], np.flatnonzero(np.diff(row)) + 1, [64]])
                runs += int((np.diff(cuts) >= 3).sum())
            most = max(most, runs)
    return most


@pytest.mark.parametrize("cell, cells, least", [(32.0, 28, 65), (20.0, 40, 100)])
def test_tiles_of_many_planes_match_the_oracle(oracle, monkeypatch, cell, cells, least):
    from gradoom_amd import hostmath, mapbuild, synthmap
    from gradoom_amd.renderer import HipRenderer, LaneState
    from gradoom_amd.selfcheck import make_lane_arrays

    monkeypatch.setattr(synthmap, "CELL", cell)       # small sectors, each a step of a few units from its neighbours
    monkeypatch.setattr(synthmap, "JITTER", 3)
    cosine = hostmath.cosine_correction("cpu").numpy()
    smap = synthmap.generate_map(91, grid=(cells, cells), sectors=cells * cells, linedefs=2 * cells * (cells + 1))
    rng = np.random.default_rng(5)
    smap.sector_heights[:, 0] = rng.integers(0, 4, len(smap.sector_heights))
    smap.sector_heights[:, 1] = 180 + rng.integers(0, 4, len(smap.sector_heights))
    poses = synthmap.generate_poses(smap, LANES, 93)
    poses.view_z[:] = [20, 41, 60, 90, 120, 41]
    arrays = make_lane_arrays(smap, poses, synthmap.generate_sprites(smap, LANES, 4, 94))
    tables = mapbuild.build_map_tables(smap)
    result = oracle.render(tables, arrays, cosine, debug_lane=2)
    assert _runs(result["debug"]["scene_depth"]) >= least
    renderer = HipRenderer(smap, LANES, "cuda:0", cosine_correction=cosine, tables=tables)
    for offset in (0, 1):                             # frames on a word, and on no word
        indexed = torch.zeros(LANES * 240 * 320 + offset, dtype=torch.uint8, device="cuda:0")[offset:].view(LANES, 240, 320)
        renderer.scribble(0xA5)
        renderer.render(LaneState.from_numpy(arrays, "cuda:0"), indexed=indexed)
        torch.cuda.synchronize()
        assert renderer.status() == 0
        assert np.array_equal(indexed.cpu().numpy(), result["indexed"]), offset
    renderer.close()
