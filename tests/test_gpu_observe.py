"""The pooling kernel where its work-groups take one block of rows, several, or blocks of two frames, and on frames that start on any byte."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _weights(out_size: int, in_size: int, unit: int) -> torch.Tensor:
    low = lambda k, size: k * size  # noqa: E731
    out, inner = torch.arange(out_size)[:, None], torch.arange(in_size)[None, :]
    end = torch.minimum(low(out + 1, in_size), low(inner + 1, out_size))
    start = torch.maximum(low(out, in_size), low(inner, out_size))
    return ((end - start).clamp(min=0) // unit).to(torch.float64)


def _pooled(indexed: torch.Tensor, palette: torch.Tensor) -> torch.Tensor:
    """In whole numbers, which float64 holds: rows and columns weighted by their overlaps, rounded per channel, then the grey level."""
    black = torch.zeros((indexed.shape[0], 240 - indexed.shape[1], 320, 3), dtype=torch.float64)
    colours = torch.cat([palette[indexed.long()].to(torch.float64), black], dim=1)
    sums = torch.tensordot(torch.tensordot(_weights(84, 240, 12), colours, ([1], [1])), _weights(84, 320, 4), ([2], [1]))   # [84, N, 3, 84]
    channels = ((sums.permute(1, 0, 3, 2).to(torch.int64) + 800) // 1600)
    return ((channels * torch.tensor([77, 150, 29])).sum(3) + 128 >> 8).to(torch.uint8)


@pytest.mark.parametrize("lanes", [1, 2, 341, 342, 700])   # 1023 and 1026 blocks of rows: the line where a work-group gets more than one
@pytest.mark.parametrize("rows", [208, 240])
@pytest.mark.parametrize("offset", [0, 4, 1])
def test_pooled_frames_equal_the_weighted_sums(lanes, rows, offset):
    from gradoom_amd import ops

    generator = torch.Generator().manual_seed(lanes * 1000 + rows + offset)
    palette = torch.randint(0, 256, (256, 3), generator=generator, dtype=torch.uint8)
    palette[:2] = torch.tensor([[0, 0, 0], [255, 255, 255]], dtype=torch.uint8)
    frames = torch.randint(0, 256, (lanes, rows, 320), generator=generator, dtype=torch.uint8)
    frames[0] = 1                         # the largest sums there are
    if lanes > 1:
        frames[1] = 0
    held = torch.zeros(offset + frames.numel(), dtype=torch.uint8, device="cuda:0")
    indexed = held[offset:].view(frames.shape)
    indexed.copy_(frames)
    got = ops.policy_area_grayscale(indexed, palette.to("cuda:0")).cpu()
    for first in range(0, lanes, 64):
        assert torch.equal(got[first:first + 64], _pooled(frames[first:first + 64], palette))


CAMERAS = 5


def _blended(palette: np.ndarray, bonus: np.float32, flash: np.float32) -> np.ndarray:
    """engine.py:15385-15397, a rounded float32 operation at a time."""
    one, gold, red = np.float32(1), np.array([215, 186, 69], dtype=np.float32), np.array([255, 0, 0], dtype=np.float32)
    value = palette.astype(np.float32) * (one - bonus) + gold * bonus
    return np.clip(value * (one - flash) + red * flash, 0, 255).astype(np.uint8)


# both sides of the line where a work-group takes half a block of rows and no more; of that where it takes several blocks, which end one lane and begin the next
@pytest.mark.parametrize("lanes", [1, "the last few", "the first that are more", 341, 342, 700, 1030])
@pytest.mark.parametrize("layout, rows, masked", [("chw", 208, False), ("hwc", 240, False), ("chw", 240, True)])
def test_stacks_of_lanes_that_flash_differently_match_the_oracle(oracle, lanes, layout, rows, masked):
    """A palette of its own a lane, stacks that roll or are filled anew by a mask, and their copies."""
    import launch_rules
    from gradoom_amd import hostmath, mapbuild
    from gradoom_amd.renderer import HipRenderer, LaneState
    from gradoom_amd.selfcheck import make_lane_arrays
    from random_cases import closed_door_parts

    if isinstance(lanes, str):
        (line,) = launch_rules.lines("observe_few")
        lanes = line - 1 if lanes == "the last few" else line
    cosine = hostmath.cosine_correction("cpu").numpy()
    smap, poses, sprites, styles = closed_door_parts(6002, CAMERAS, mixed=True)
    arrays = make_lane_arrays(smap, poses, sprites)
    arrays["sprite_style"] = styles
    tables = mapbuild.build_map_tables(smap)
    rng = np.random.default_rng(lanes)
    arrays["screen_blend"] = rng.random((CAMERAS, 2), dtype=np.float32)
    drawn = oracle.render(tables, arrays, cosine, obs_source_rows=rows)
    which = np.arange(lanes) % CAMERAS
    arrays = {name: np.ascontiguousarray(value[which]) for name, value in arrays.items()}
    arrays["screen_blend"][CAMERAS:] = rng.random((max(lanes - CAMERAS, 0), 2), dtype=np.float32)
    palette = np.asarray(tables["playpal"], dtype=np.uint8).reshape(256, 3)
    expected = np.concatenate([oracle.observe(drawn["indexed"][which[n]][None, :rows], _blended(palette, *arrays["screen_blend"][n]))[0] for n in range(lanes)])
    assert np.array_equal(expected[:CAMERAS], drawn["obs"][:lanes])
    old = rng.integers(0, 256, (lanes, 4, 84, 84), dtype=np.uint8)
    mask = rng.random(lanes) < 0.4
    filled = np.repeat(expected[:, None], 4, axis=1)
    rolled = old if masked else np.concatenate((old[:, 1:], expected[:, None]), axis=1)
    stacks = np.where(mask[:, None, None, None], filled, rolled)
    to = lambda value: torch.as_tensor(value, device="cuda:0")  # noqa: E731
    obs, frames = torch.zeros((lanes, 84, 84), dtype=torch.uint8, device="cuda:0"), to(old)
    final = torch.zeros((lanes, 4, 84, 84) if layout == "chw" else (lanes, 84, 84, 4), dtype=torch.uint8, device="cuda:0")
    renderer = HipRenderer(smap, lanes, "cuda:0", cosine_correction=cosine, tables=tables)
    renderer.render(LaneState.from_numpy(arrays, "cuda:0"), obs=obs, frames=frames, reset_mask=to(mask), stack_only_masked=masked, final_frames=final, final_layout=layout, obs_source_rows=rows)
    torch.cuda.synchronize()
    assert renderer.status() == 0
    renderer.close()
    assert np.array_equal(obs.cpu().numpy(), expected)
    assert np.array_equal(frames.cpu().numpy(), stacks)
    assert np.array_equal((final if layout == "chw" else final.permute(0, 3, 1, 2)).cpu().numpy(), stacks)
