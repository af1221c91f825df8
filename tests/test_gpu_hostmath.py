"""The library's ray tables and billboard depths against the Torch expressions they replace, bit for bit."""

from __future__ import annotations

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lanes, slots", [(1, 1), (3, 85), (257, 7), (4096, 1)])
def test_ray_tables_and_sprite_depths_have_the_bits_of_the_torch_expressions(lanes, slots):
    from gradoom_amd import hostmath

    device = "cuda:0"
    generator = torch.Generator(device=device).manual_seed(lanes)
    rand = lambda *shape: torch.rand(shape, generator=generator, device=device)  # noqa: E731
    angle = rand(lanes) * 2 * math.pi
    x, y = rand(lanes) * 6000 - 3000, rand(lanes) * 6000 - 3000
    sprite_x, sprite_y = x[:, None] + rand(lanes, slots) * 400 - 200, y[:, None] + rand(lanes, slots) * 400 - 200
    sprite_x[0, 0], sprite_y[0, 0] = x[0], y[0]              # at the eye
    angle[-1] = -0.0
    offsets = hostmath.native_ray_offsets(device)
    print(f"{lanes} lanes, {slots} billboards", flush=True)
    ray_cos, ray_sin = hostmath.ray_tables(angle, offsets)
    rays = angle[:, None] + offsets[None, :]
    assert torch.equal(ray_cos.view(torch.int32), torch.cos(rays).view(torch.int32)) and torch.equal(ray_sin.view(torch.int32), torch.sin(rays).view(torch.int32))
    dx, dy = sprite_x - x[:, None], sprite_y - y[:, None]
    relative = torch.remainder(torch.atan2(dy, dx) - angle[:, None] + math.pi, 2 * math.pi) - math.pi
    expected = torch.sqrt(dx * dx + dy * dy).clamp_min(1) * torch.cos(relative)
    depth = hostmath.sprite_depth(x, y, angle, sprite_x, sprite_y)
    assert torch.equal(depth.view(torch.int32), expected.view(torch.int32))
    together = hostmath.lane_floats_kernel(x, y, angle, offsets, sprite_x, sprite_y)
    assert all(torch.equal(one.view(torch.int32), other.view(torch.int32)) for one, other in zip(together, (ray_cos, ray_sin, depth)))
