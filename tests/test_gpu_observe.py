"""The pooling kernel where its work-groups take one block of rows, several, or blocks of two frames, and on frames that start on any byte."""

from __future__ import annotations

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
