"""The vector environment's kernels against the Torch expressions they stand in for, at lane counts around the edges of their work-groups."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import load_fixture

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lanes, sprites", [(1, 0), (63, 5), (257, 129), (1025, 1)])
def test_pose_pool_and_bookkeeping_equal_the_torch_expressions(lanes, sprites):
    from gradoom_amd.env import GraDoomVecEnv, PosePoolDynamics

    _meta, _data, smap, _tables = load_fixture("tiny_stages")

    class NoRenderer:
        def render(self, *_args, **_kwargs):
            pass

    envs = []
    for device in ("cuda:0", "cpu"):   # on the CPU everything takes the Torch expressions
        dynamics = PosePoolDynamics(smap, lanes, device, pool=7, sprites=sprites, episode_timeout=3, seed=5)
        envs.append(GraDoomVecEnv(smap, lanes, device=device, dynamics=dynamics, renderer=NoRenderer()))
    generator = torch.Generator().manual_seed(lanes)
    ints = lambda low, high: torch.randint(low, high, (lanes,), generator=generator)  # noqa: E731
    masks = [torch.ones(lanes, dtype=torch.bool), ints(0, 2).bool()]
    print(f"{lanes} lanes, {sprites} billboards", flush=True)
    for mask in masks:
        seeds = ints(-(1 << 40), 1 << 40)
        for env in envs:
            env.reset_device(mask.to(env.device), seeds.to(env.device))
    for step in range(4):
        actions, seeds = ints(-9, 17), ints(0, 1 << 31)
        with_reset = step >= 2
        outs = []
        for env in envs:
            call = (actions.to(env.device), seeds.to(env.device))
            outs.append(env.step_and_reset_device(*call) if with_reset else env.step_device(call[0]))
        for name in ("rewards", "terminated", "truncated", "signals") + (("final_signals",) if with_reset else ()):
            assert torch.equal(getattr(outs[0], name).cpu(), getattr(outs[1], name)), name
        for name in ("pending_reset", "_initialized", "_latest_reset_seeds", "signal_buffer"):
            assert torch.equal(getattr(envs[0], name).cpu(), getattr(envs[1], name)), name
        ours, theirs = (env._dynamics.lane_state() for env in envs)
        for name, value in vars(theirs).items():
            assert (value is None) == (getattr(ours, name) is None), name
            assert value is None or torch.equal(getattr(ours, name).cpu(), value), name
    rows = torch.arange(0, lanes, 2)
    ours, theirs = envs[0]._dynamics.lane_state(rows.to("cuda:0")), envs[1]._dynamics.lane_state(rows)
    assert torch.equal(ours.x.cpu(), theirs.x) and torch.equal(ours.angle_bam.cpu(), theirs.angle_bam)
    for bad in (17, -1):
        actions = torch.zeros(lanes, dtype=torch.int64)
        actions[-1] = bad
        envs[0].pending_reset.zero_()
        with pytest.raises(ValueError, match="outside the declared action space"):
            envs[0].step(actions.to("cuda:0"))


@pytest.mark.parametrize("lanes, rows", [(1, 1), (1, 208), (3, 240), (2, 7)])
def test_rgb_expansion_in_device_and_pinned_memory(lanes, rows):
    from gradoom_amd.renderer import HipRenderer

    _meta, _data, smap, tables = load_fixture("tiny_stages")
    renderer = HipRenderer(smap, 1, "cuda:0", tables=tables)
    generator = torch.Generator(device="cuda:0").manual_seed(rows)
    indexed = torch.randint(0, 256, (lanes, rows, 320), generator=generator, device="cuda:0", dtype=torch.uint8)
    guarded = torch.full((lanes * rows * 960 + 64,), 7, dtype=torch.uint8, device="cuda:0")
    print(f"{lanes} x {rows} rows", flush=True)
    for offset in (0, 1):              # the second not aligned to the sixteen bytes of a store
        guarded.fill_(7)
        rgb = guarded[offset : offset + lanes * rows * 960].view(lanes, rows, 320, 3)
        renderer.expand_rgb24(indexed, rgb)
        assert np.array_equal(rgb.cpu().numpy(), np.asarray(tables["playpal"])[indexed.cpu().numpy()])
        assert bool((guarded[offset + lanes * rows * 960 :] == 7).all())
    renderer.close()


@pytest.mark.parametrize("part", [1, 2, 4, 5, 6, 2**31 - 1])   # five frames; the last stands for any number beyond them
def test_rgb_frames_by_parts_of_any_size(part):
    import ctypes

    from gradoom_amd.renderer import HipRenderer

    _meta, _data, smap, tables = load_fixture("tiny_stages")
    renderer = HipRenderer(smap, 1, "cuda:0", tables=tables)
    indexed = torch.randint(0, 256, (5, 240, 320), generator=torch.Generator(device="cuda:0").manual_seed(part), device="cuda:0", dtype=torch.uint8)
    staging, frames = torch.zeros((5, 240, 320, 3), dtype=torch.uint8, pin_memory=True), np.zeros((5, 240, 320, 3), dtype=np.uint8)
    print(f"parts of {part}", flush=True)
    renderer.expand_rgb_to_pieces(indexed, staging, part, (ctypes.c_void_p * 5)(*[frame.ctypes.data for frame in frames]))
    assert np.array_equal(frames, np.asarray(tables["playpal"])[indexed.cpu().numpy()])
    renderer.close()


@pytest.mark.parametrize("form", ["int64", "int32", "strided", "two_dimensions", "list", "negative", "none"])
def test_the_lanes_asked_of_a_pose_pool_may_come_in_any_form(form):
    """A kernel reads int64 rows of one contiguous piece; whatever else is handed in goes the way of the Torch expressions."""
    from gradoom_amd.env import PosePoolDynamics

    _meta, _data, smap, _tables = load_fixture("tiny_stages")
    pools = [PosePoolDynamics(smap, 9, device, pool=7, sprites=3, seed=5) for device in ("cuda:0", "cpu")]
    rows = torch.tensor([8, 1, 1, 0, 5, 3])
    rows = {"int64": rows, "int32": rows.to(torch.int32), "strided": torch.stack([rows, rows.flip(0)], 1)[:, 1], "two_dimensions": rows.view(2, 3),
            "list": rows.tolist(), "negative": rows - 9, "none": rows[:0]}[form]
    for pool in pools:
        pool.reset(torch.ones(9, dtype=torch.bool, device=pool.device), torch.arange(9, device=pool.device))
    on_device = rows if isinstance(rows, list) else rows.to("cuda:0")
    if form == "strided":
        on_device = torch.stack([on_device, on_device], 1)[:, 0]
        assert not on_device.is_contiguous()
    print(form, flush=True)
    ours, theirs = pools[0].lane_state(on_device), pools[1].lane_state(rows)
    for name, value in vars(theirs).items():
        assert value is None or torch.equal(getattr(ours, name).cpu(), value), name
