"""Float32 transcendentals the renderer takes as inputs, computed with Torch.

The reference evaluates a handful of ``cos/sin/atan/atan2/sqrt`` expressions
with Torch ops on the engine's device; their bit patterns are a property of the
Torch build, not of the algorithm.  The kernels therefore receive these values
as inputs, produced here by the very same Torch expressions on whichever device
the lane tensors live on:

* ``native_ray_offsets = -atan((x - 160) / 160)``      (``engine.py:2050-2054``)
* ``cosine_correction  = cos(native_ray_offsets)``      (``engine.py:10967``)
* ``ray_cos/ray_sin    = cos/sin(angle + offsets)``     (``engine.py:10966-10974``)
* ``sprite depth       = clamp_min(sqrt(dx²+dy²),1) * cos(wrap(atan2(dy,dx) - angle))``
  (``engine.py:14684-14688``)
* retained view angle ``bam.float() * (2π / 2³²)``      (``engine.py:10651``)

Tensors on a ROCm device take one kernel of the library for the ray tables and one for the sprite depths, which
give the Torch expressions' bits (``gd_ray_tables``, ``gd_sprite_depth``); everything else takes the expressions, and so
does a call that Torch records, transforms or traces (a gradient, ``vmap``, forward mode, ``torch.compile``, fake tensors).
"""

from __future__ import annotations

import math

import torch
from torch.autograd import forward_ad
from torch.utils._device import DeviceContext

SCREEN_WIDTH = 320
BAM_TO_RADIANS = 2.0 * math.pi / float(1 << 32)


def native_ray_offsets(device) -> torch.Tensor:
    columns = torch.arange(SCREEN_WIDTH, device=device, dtype=torch.float32) - SCREEN_WIDTH / 2.0
    return -torch.atan(columns / (SCREEN_WIDTH / 2.0))


def cosine_correction(device) -> torch.Tensor:
    return torch.cos(native_ray_offsets(device))


def _plain_call(*tensors: torch.Tensor) -> bool:
    """Does this call want the values of these tensors and nothing else: is nothing recorded, transformed or traced?"""

    if torch.compiler.is_compiling() or torch._C._get_tracing_state() is not None:
        return False
    if torch._C._functorch.peek_interpreter_stack() is not None or forward_ad._current_level >= 0:   # vmap, grad, jvp; dual numbers
        return False
    if torch._C._len_torch_dispatch_stack() > 0:                                                     # fake tensors, make_fx
        return False
    if torch._C._len_torch_function_stack() > 0 and any(type(mode) is not DeviceContext for mode in torch.overrides._get_current_function_mode_stack()):
        return False                                                                                 # (torch.set_default_device is no matter)
    recorded = torch.is_grad_enabled()
    for tensor in tensors:
        if type(tensor) is not torch.Tensor or tensor.is_neg() or (recorded and tensor.requires_grad):
            return False
    return True


def _on_device(*tensors: torch.Tensor) -> bool:
    """Are these contiguous float32 tensors of one ROCm device, as the library's kernels read them, and is only their result wanted?"""

    device = tensors[0].device
    if device.type != "cuda" or not _plain_call(*tensors):
        return False
    for tensor in tensors:
        if tensor.dtype is not torch.float32 or tensor.device != device or not tensor.is_contiguous():
            return False
    return True


def ray_tables_kernel(angle: torch.Tensor, offsets: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    """``ray_tables`` of tensors that are known to be what the kernel reads (``[N]`` and ``[320]``), by the kernel."""

    from . import _lib  # noqa: PLC0415

    tables = torch.empty((2, angle.shape[0], SCREEN_WIDTH), dtype=torch.float32, device=angle.device)
    ray_cos, ray_sin = tables[0], tables[1]
    with torch.cuda.device(angle.device):
        _lib.check(_lib.library().gd_ray_tables(angle.data_ptr(), offsets.data_ptr(), angle.shape[0], ray_cos.data_ptr(), ray_sin.data_ptr(),
                                                torch.cuda.current_stream(angle.device).cuda_stream))
    return ray_cos, ray_sin


def ray_tables(angle: torch.Tensor, offsets: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    if _on_device(angle, offsets) and angle.dim() == 1 and offsets.shape == (SCREEN_WIDTH,):
        return ray_tables_kernel(angle, offsets)
    ray_angles = angle[:, None] + offsets[None, :]
    return torch.cos(ray_angles).contiguous(), torch.sin(ray_angles).contiguous()


def angle_from_bam(angle_bam: torch.Tensor) -> torch.Tensor:
    return angle_bam.to(torch.float32) * BAM_TO_RADIANS


def sprite_depth_kernel(x, y, angle, sprite_x, sprite_y) -> torch.Tensor:
    """``sprite_depth`` of tensors that are known to be what the kernel reads (``[N]`` three times, ``[N, A]`` twice), by the kernel."""

    from . import _lib  # noqa: PLC0415

    depth = torch.empty_like(sprite_x)
    with torch.cuda.device(x.device):
        _lib.check(_lib.library().gd_sprite_depth(x.data_ptr(), y.data_ptr(), angle.data_ptr(), sprite_x.data_ptr(), sprite_y.data_ptr(), sprite_x.shape[0],
                                                  sprite_x.shape[1], depth.data_ptr(), torch.cuda.current_stream(x.device).cuda_stream))
    return depth


def lane_floats_kernel(x, y, angle, offsets, sprite_x, sprite_y) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """``ray_tables_kernel`` and ``sprite_depth_kernel`` in one launch: (ray_cos, ray_sin, depth)."""

    from . import _lib  # noqa: PLC0415

    count, slots = sprite_x.shape
    rays = count * SCREEN_WIDTH
    floats = torch.empty(2 * rays + count * slots, dtype=torch.float32, device=angle.device)
    ray_cos, ray_sin, depth = floats[:rays].view(count, SCREEN_WIDTH), floats[rays : 2 * rays].view(count, SCREEN_WIDTH), floats[2 * rays :].view(count, slots)
    with torch.cuda.device(angle.device):
        _lib.check(_lib.library().gd_lane_floats(x.data_ptr(), y.data_ptr(), angle.data_ptr(), offsets.data_ptr(), sprite_x.data_ptr(), sprite_y.data_ptr(), count, slots,
                                                 ray_cos.data_ptr(), ray_sin.data_ptr(), depth.data_ptr(), torch.cuda.current_stream(angle.device).cuda_stream))
    return ray_cos, ray_sin, depth


def sprite_depth(x, y, angle, sprite_x, sprite_y) -> torch.Tensor:
    if _on_device(x, y, angle, sprite_x, sprite_y) and x.shape == y.shape == angle.shape == sprite_x.shape[:1] and sprite_x.shape == sprite_y.shape and sprite_x.dim() == 2:
        return sprite_depth_kernel(x, y, angle, sprite_x, sprite_y)
    dx = sprite_x - x[:, None]
    dy = sprite_y - y[:, None]
    distance = torch.sqrt(dx * dx + dy * dy).clamp_min(1)
    relative = torch.remainder(torch.atan2(dy, dx) - angle[:, None] + math.pi, 2 * math.pi) - math.pi
    return (distance * torch.cos(relative)).contiguous()
