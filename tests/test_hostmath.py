"""Which calls of the float32 helpers may leave Torch for a kernel of the library (CPU only), and what the others compute."""

from __future__ import annotations

import math

import pytest
import torch
from torch.autograd import forward_ad


def _calls():
    """How a call can be more than its values: each hands ``ask`` the tensors as a helper would get them."""

    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    class Counting(TorchDispatchMode):
        def __torch_dispatch__(self, func, _types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Watching(TorchFunctionMode):
        def __torch_function__(self, func, _types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Named(torch.Tensor):
        pass

    def under(mode, ask):
        with mode:
            ask(torch.zeros(3))

    def dual(ask):
        with forward_ad.dual_level():
            ask(forward_ad.make_dual(torch.zeros(3), torch.ones(3)))

    def mapped(ask):
        torch.vmap(lambda x: (ask(x), x)[1])(torch.zeros(2, 3))

    def gradient(ask):
        torch.func.grad(lambda x: (ask(x), x.sum())[1])(torch.zeros(3))

    def traced(ask):
        torch.jit.trace(lambda x: (ask(x), x + 1)[1], (torch.zeros(3),), check_trace=False)

    return {
        "requires_grad": lambda ask: ask(torch.zeros(3, requires_grad=True)), "dual": dual, "vmap": mapped, "grad": gradient,
        "jit_trace": traced, "fake": lambda ask: under(FakeTensorMode(), ask), "make_fx": lambda ask: make_fx(lambda x: (ask(x), x + 1)[1])(torch.zeros(3)),
        "dispatch_mode": lambda ask: under(Counting(), ask), "function_mode": lambda ask: under(Watching(), ask),
        "subclass": lambda ask: ask(torch.zeros(3).as_subclass(Named)), "negative": lambda ask: ask(torch._neg_view(torch.zeros(3))),
    }


@pytest.mark.parametrize("how", ["requires_grad", "dual", "vmap", "grad", "jit_trace", "fake", "make_fx", "dispatch_mode", "function_mode", "subclass", "negative"])
def test_a_call_that_torch_records_transforms_or_traces_stays_in_torch(how):
    from gradoom_amd import hostmath

    answers = []
    _calls()[how](lambda *tensors: answers.append(hostmath._plain_call(*tensors)))
    assert answers and not any(answers)


def test_an_ordinary_call_is_a_plain_one():
    from gradoom_amd import hostmath

    wants_grad = torch.zeros(3, requires_grad=True)
    assert hostmath._plain_call(torch.zeros(3), torch.ones(2, 2))
    with torch.no_grad():
        assert hostmath._plain_call(wants_grad)
    with torch.inference_mode():
        assert hostmath._plain_call(torch.zeros(3))
    with torch.device("cpu"):       # what torch.set_default_device leaves in place
        assert hostmath._plain_call(torch.zeros(3))


@pytest.mark.gpu
def test_gradients_vmap_and_forward_mode_go_through_on_the_device():
    from gradoom_amd import hostmath

    device = "cuda:0"
    generator = torch.Generator(device=device).manual_seed(7)
    angle = torch.rand(5, generator=generator, device=device) * 2 * math.pi
    offsets = hostmath.native_ray_offsets(device)
    wants_grad = angle.clone().requires_grad_()
    ray_cos, ray_sin = hostmath.ray_tables(wants_grad, offsets)
    ray_cos.sum().backward()
    assert torch.allclose(wants_grad.grad, -torch.sin(angle[:, None] + offsets).sum(1), rtol=1e-5, atol=1e-4)   # 320 terms of one unit: 320 * 2^-24 each way
    plain = hostmath.ray_tables(angle, offsets)
    assert torch.equal(ray_cos, plain[0]) and torch.equal(ray_sin, plain[1])
    mapped = torch.vmap(lambda a: torch.stack(hostmath.ray_tables(a, offsets)))(angle[:4].view(2, 2))
    assert torch.equal(mapped[1], torch.stack(hostmath.ray_tables(angle[2:4], offsets)))
    x, y = angle * 100, angle * 70
    sprites = torch.rand(2, 5, 3, generator=generator, device=device) * 500
    with forward_ad.dual_level():
        depth = hostmath.sprite_depth(forward_ad.make_dual(x, torch.ones_like(x)), y, angle, sprites[0], sprites[1])
        value, tangent = forward_ad.unpack_dual(depth)
        assert tangent is not None and bool(tangent.abs().sum() > 0)
    assert torch.equal(value, hostmath.sprite_depth(x, y, angle, sprites[0], sprites[1]))
