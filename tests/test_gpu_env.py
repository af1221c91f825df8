"""The vector-env front end on the real renderer (needs an MI355X)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import load_fixture

pytestmark = pytest.mark.gpu


def test_step_and_reset_device_matches_oracle_frame_by_frame(oracle):
    from gradoom_amd import hostmath
    from gradoom_amd.env import GraDoomVecEnv

    _meta, _data, smap, tables = load_fixture("small_midtex_sprites")
    lanes = 5
    env = GraDoomVecEnv(smap, lanes, device="cuda:0", render_mode="rgb_array", episode_timeout=2, sprites=16)
    cosine = env._renderer._cosine   # the renderer's own table (the GPU's float32 cosines, like its ray tables)

    def expected_obs():
        state = env._dynamics.lane_state()
        arrays = {}
        for name in ("x", "y", "angle", "view_z", "x_fixed", "y_fixed", "angle_bam", "pitch_bam", "flash_light",
                     "sprite_x", "sprite_y", "sprite_z", "sprite_id", "sprite_alive", "sprite_fullbright"):
            arrays[name] = getattr(state, name).cpu().numpy()
        # the env computes the float32 tables with Torch on the GPU; hand the oracle the same values
        ray_cos, ray_sin = hostmath.ray_tables(state.angle, env._renderer.ray_offsets)
        arrays["ray_cos"], arrays["ray_sin"] = ray_cos.cpu().numpy(), ray_sin.cpu().numpy()
        arrays["sprite_depth"] = hostmath.sprite_depth(state.x, state.y, state.angle, state.sprite_x, state.sprite_y).cpu().numpy()
        return oracle.render(tables, arrays, cosine)

    mask = torch.ones(lanes, dtype=torch.bool, device="cuda:0")
    seeds = torch.arange(lanes, device="cuda:0")
    obs, _signals = env.reset_device(mask, seeds)
    first = expected_obs()
    for k in range(4):
        assert np.array_equal(obs[:, k].cpu().numpy(), first["obs"])
    actions = torch.zeros(lanes, dtype=torch.int64, device="cuda:0")
    transition = env.step_and_reset_device(actions, seeds)
    second = expected_obs()
    assert np.array_equal(transition.observations[:, 3].cpu().numpy(), second["obs"])
    assert np.array_equal(transition.observations[:, 2].cpu().numpy(), first["obs"])
    assert not bool(transition.truncated.any())
    transition = env.step_and_reset_device(actions, seeds + 7)
    assert bool(transition.truncated.all())
    third = expected_obs()   # dynamics already reset: all four stack entries show the reset frame
    for k in range(4):
        assert np.array_equal(transition.observations[:, k].cpu().numpy(), third["obs"])
    assert not np.array_equal(transition.final_observations.cpu().numpy(), transition.observations.cpu().numpy())
    image = env.render()
    assert image.shape == (240, 320, 3)
    assert np.array_equal(image, np.asarray(tables["playpal"])[third["indexed"][0]])
    assert env._renderer.status() == 0
    env.close()


def test_host_api_safe_view_buffers_are_written_by_the_renderer():
    # reset()/step() hand out two buffers in turn (env.py:459-472, 678-688); they hold the stack, in either layout
    from gradoom_amd.env import GraDoomVecEnv

    _meta, _data, smap, _tables = load_fixture("small_midtex_sprites")
    lanes = 6
    actions = torch.zeros(lanes, dtype=torch.int64, device="cuda:0")
    for layout in ("chw", "hwc"):
        env = GraDoomVecEnv(smap, lanes, device="cuda:0", episode_timeout=50, sprites=8, obs_layout=layout, obs_copy="safe_view")
        view = (lambda t: t) if layout == "chw" else (lambda t: t.permute(0, 2, 3, 1))
        first, _ = env.reset(seed=4)
        assert first.data_ptr() != env.frames.data_ptr() and torch.equal(first, view(env.frames))
        held = first.clone()
        second = env.step(actions)[0]
        assert second.data_ptr() != first.data_ptr()
        assert torch.equal(first, held) and torch.equal(second, view(env.frames))
        assert not torch.equal(first, second)
        third = env.step(actions)[0]
        assert third.data_ptr() == first.data_ptr() and torch.equal(third, view(env.frames))
        env.close()


def test_more_than_256_linedefs_in_one_column_raise_in_the_environment(monkeypatch):
    # A corridor of 300 narrow sectors seen end on: every divider lands in the same few screen columns, more than the 256
    # candidates a column can hold in the spill pool (64 in its own slots).  The environment must say so rather than hand
    # out the frame.
    from gradoom_amd import synthmap
    from gradoom_amd.env import GraDoomVecEnv, PosePoolDynamics

    monkeypatch.setattr(synthmap, "CELL", 48)   # 300 cells of the usual 256 units would leave the 16.16 coordinate range
    smap = synthmap.generate_map(5, grid=(300, 1), sectors=300, linedefs=901)
    lanes = 2
    dynamics = PosePoolDynamics(smap, lanes, "cuda:0", pool=4)
    quad = smap.sector_quads[0]
    centre = quad.mean(axis=0)
    dynamics._pool["x"].fill_(float(centre[0]))
    dynamics._pool["y"].fill_(float(centre[1]))
    dynamics._pool["angle_bam"].zero_()       # looking along +x, down the corridor
    dynamics._pool["pitch_bam"].zero_()
    dynamics._pool["view_z"].fill_(float(smap.sector_heights[0, 0]) + 41.0)
    env = GraDoomVecEnv(smap, lanes, device="cuda:0", dynamics=dynamics, render_mode="rgb_array")
    mask = torch.ones(lanes, dtype=torch.bool, device="cuda:0")
    env.reset_device(mask, torch.arange(lanes, device="cuda:0"))
    assert env._renderer.status() & 1
    with pytest.raises(RuntimeError, match="truncated a screen column's candidate list"):
        env.step_and_reset_device(torch.zeros(lanes, dtype=torch.int64, device="cuda:0"), torch.arange(lanes, device="cuda:0"))
    with pytest.raises(RuntimeError, match="truncated"):
        env.render()
    with pytest.raises(RuntimeError, match="truncated"):
        env.close()
    assert env.closed


def test_a_step_does_not_wait_for_other_streams():
    from gradoom_amd.env import GraDoomVecEnv

    _meta, _data, smap, _tables = load_fixture("tiny_stages")
    lanes = 3
    env = GraDoomVecEnv(smap, lanes, device="cuda:0", episode_timeout=2)
    env.reset_device(torch.ones(lanes, dtype=torch.bool, device="cuda:0"), torch.arange(lanes, device="cuda:0"))
    actions, seeds = torch.zeros(lanes, dtype=torch.int64, device="cuda:0"), torch.arange(lanes, device="cuda:0")
    for _ in range(4):
        env.step_and_reset_device(actions, seeds)
    # a kernel of some 50 ms on another stream; streams share a few hardware queues, so one of several must do
    started, ended = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    cycles = 100_000
    torch.cuda._sleep(cycles)
    started.record()
    torch.cuda._sleep(cycles)
    ended.record()
    torch.cuda.synchronize()
    cycles = int(cycles * 50.0 / max(started.elapsed_time(ended), 0.01))
    still_running = 0
    for stream in [torch.cuda.Stream() for _ in range(6)]:
        with torch.cuda.stream(stream):
            torch.cuda._sleep(cycles)
            ended.record()
        env.step_and_reset_device(actions, seeds)
        still_running += not ended.query()
        torch.cuda.synchronize()
    print(f"{still_running} of 6 steps ended before the other stream's kernel", flush=True)
    assert still_running > 0
    assert env._renderer.status_seen() == env._renderer.status() == 0
    env.close()


@pytest.mark.parametrize("timeout", [1, 50])
def test_a_step_with_truncated_frames_is_refused_whether_lanes_end_or_not(monkeypatch, timeout):
    """The reset of the lanes that end is queued behind the step's frames, which the host does not wait for: their check comes all the same."""

    from gradoom_amd.env import GraDoomVecEnv

    _meta, _data, smap, _tables = load_fixture("small_midtex_sprites")
    lanes = 3
    env = GraDoomVecEnv(smap, lanes, device="cuda:0", episode_timeout=timeout, sprites=4)
    actions, seeds = torch.zeros(lanes, dtype=torch.int64, device="cuda:0"), torch.arange(lanes, device="cuda:0")
    env.reset_device(torch.ones(lanes, dtype=torch.bool, device="cuda:0"), seeds)
    assert bool(env.step_and_reset_device(actions, seeds).truncated.all()) == (timeout == 1)
    monkeypatch.setattr(env._renderer, "status_seen", lambda: 1)
    with pytest.raises(RuntimeError, match="candidate list"):
        env.step_and_reset_device(actions, seeds)
    monkeypatch.undo()
    env.step_and_reset_device(actions, seeds)
    env.close()


@pytest.mark.parametrize("lanes", [3, 5, 113])     # frames that stay on one stream, that go to the side stream and back
def test_a_refused_step_has_reset_no_lane(monkeypatch, lanes):
    """Every lane ends with the step whose frames are truncated: the lanes, their stacks and seeds stay as the step left them, and bad seeds are not
    what the step is refused for."""

    from gradoom_amd.env import GraDoomVecEnv

    _meta, _data, smap, _tables = load_fixture("small_midtex_sprites")
    envs = [GraDoomVecEnv(smap, lanes, device="cuda:0", episode_timeout=2, sprites=4) for _ in range(2)]
    actions, seeds = torch.zeros(lanes, dtype=torch.int64, device="cuda:0"), torch.arange(lanes, device="cuda:0") + 7
    for env in envs:
        env.reset_device(torch.ones(lanes, dtype=torch.bool, device="cuda:0"), seeds)
        env.step_and_reset_device(actions, seeds + 1)
    envs[1].step_device(actions)
    monkeypatch.setattr(envs[0]._renderer, "status_seen", lambda: 1)
    with pytest.raises(RuntimeError, match="candidate list"):
        envs[0].step_and_reset_device(actions, seeds[:1].float())
    monkeypatch.undo()
    states = [(env.pending_reset, env._dynamics.episode_time, env._dynamics.phase, env._latest_reset_seeds, env.frames, env.signal_buffer) for env in envs]
    assert bool(states[0][0].all()) and bool((states[0][1] == 2).all()) and torch.equal(states[0][3], seeds)
    assert all(torch.equal(one, other) for one, other in zip(*states))
    for env in envs:
        env.reset_device(torch.ones(lanes, dtype=torch.bool, device="cuda:0"), seeds)
        env.close()


@pytest.mark.parametrize("lanes", [2, 24])     # frames that stay on one stream, that go to the side stream and back
def test_the_status_is_final_where_the_frames_say_so(monkeypatch, lanes):
    """More dividers in a column than its list holds; with and without a mark, asked on the frames' own stream and on another."""

    from gradoom_amd import synthmap
    from gradoom_amd.env import PosePoolDynamics
    from gradoom_amd.renderer import HipRenderer

    monkeypatch.setattr(synthmap, "CELL", 48)
    smap = synthmap.generate_map(5, grid=(300, 1), sectors=300, linedefs=901)
    dynamics = PosePoolDynamics(smap, lanes, "cuda:0", pool=4, sprites=4)
    centre = smap.sector_quads[0].mean(axis=0)
    for name, value in (("x", float(centre[0])), ("y", float(centre[1])), ("angle_bam", 0), ("pitch_bam", 0), ("view_z", float(smap.sector_heights[0, 0]) + 41.0)):
        dynamics._pool[name].fill_(value)       # looking along +x, down the corridor
    state, obs = dynamics.lane_state(), torch.empty((lanes, 84, 84), dtype=torch.uint8, device="cuda:0")
    for marked, asked_elsewhere in ((True, False), (False, False), (True, True)):
        renderer = HipRenderer(smap, lanes, "cuda:0")
        torch.cuda.synchronize()
        renderer.wait_status()
        assert renderer.status_seen() == 0
        if marked:
            renderer.mark_status()
        renderer.render(state, obs=obs)
        stream = torch.cuda.Stream() if asked_elsewhere else torch.cuda.current_stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            renderer.wait_status()
        assert renderer.status_seen() == 1
        assert renderer.status() == 1
        renderer.close()


def test_a_pose_pool_whose_lane_state_takes_no_lanes_resets_the_lanes_that_end():
    from gradoom_amd.env import GraDoomVecEnv, PosePoolDynamics

    class Lifted(PosePoolDynamics):
        def lane_state(self):
            state = super().lane_state()
            state.view_z = state.view_z + 7.0
            return state

    _meta, _data, smap, _tables = load_fixture("tiny_stages")
    lanes = 5
    env = GraDoomVecEnv(smap, lanes, device="cuda:0", dynamics=Lifted(smap, lanes, "cuda:0", pool=7, episode_timeout=3))
    env.reset_device(torch.ones(lanes, dtype=torch.bool, device="cuda:0"), torch.arange(lanes, device="cuda:0"))
    actions, seeds = torch.zeros(lanes, dtype=torch.int64, device="cuda:0"), torch.arange(lanes, 0, -1, device="cuda:0")
    env._dynamics.episode_time[3:] = 2       # two lanes end in the next step
    transition = env.step_and_reset_device(actions, seeds)
    assert transition.truncated.tolist() == [False, False, False, True, True]
    obs = torch.zeros((lanes, 84, 84), dtype=torch.uint8, device="cuda:0")
    env._renderer.render(env._dynamics.lane_state(), obs=obs)
    for lane in (3, 4):
        assert all(torch.equal(env.frames[lane, k], obs[lane]) for k in range(4))
    assert torch.equal(env.frames[:3], transition.final_observations[:3])
    env.close()


@pytest.mark.parametrize("how", ["environment", "renderer"])
def test_a_reset_device_or_a_renderer_of_the_users_own_is_the_one_that_resets(how):
    from gradoom_amd.env import GraDoomVecEnv
    from gradoom_amd.renderer import HipRenderer

    class Counting(GraDoomVecEnv):
        resets = 0

        def reset_device(self, mask, seeds):
            self.resets += 1
            return super().reset_device(mask, seeds)

    class StackRenderer(HipRenderer):   # knows the calls that an environment made until now, and nothing of single observations
        resets = 0

        def render(self, lanes, *, frames, final_frames=None, reset_mask=None, obs=None, stack_only_masked=False, final_layout="chw"):
            assert int(lanes.x.shape[0]) == self.max_lanes and obs is None
            self.resets += reset_mask is not None
            super().render(lanes, frames=frames, final_frames=final_frames, reset_mask=reset_mask, stack_only_masked=stack_only_masked, final_layout=final_layout)

    _meta, _data, smap, _tables = load_fixture("tiny_stages")
    lanes = 3
    make = dict(device="cuda:0", episode_timeout=2)
    plain = GraDoomVecEnv(smap, lanes, **make)
    env = Counting(smap, lanes, **make) if how == "environment" else GraDoomVecEnv(smap, lanes, renderer=StackRenderer(smap, lanes, "cuda:0"), **make)
    actions, seeds = torch.zeros(lanes, dtype=torch.int64, device="cuda:0"), torch.arange(lanes, device="cuda:0")
    for each in (plain, env):
        each.reset_device(torch.ones(lanes, dtype=torch.bool, device="cuda:0"), seeds)
    for _ in range(3):               # every lane ends in the second
        ours, theirs = env.step_and_reset_device(actions, seeds), plain.step_and_reset_device(actions, seeds)
        assert torch.equal(ours.observations, theirs.observations) and torch.equal(ours.final_observations, theirs.final_observations)
    assert (env if how == "environment" else env._renderer).resets == 2
    for each in (plain, env):
        each.close()


@pytest.mark.parametrize("lanes, room", [(31, 64), (32, 64), (33, 64), (70, 48)])   # fewer than two parts, two, a part of one frame, memory for three parts
def test_rgb_frames_of_many_lanes_come_in_parts(monkeypatch, lanes, room):
    from gradoom_amd.env import GraDoomVecEnv, RGB_PART_FRAMES

    assert RGB_PART_FRAMES == 16
    monkeypatch.setattr(GraDoomVecEnv, "RGB_STAGING_BYTES", room * 240 * 320 * 3)
    _meta, _data, smap, _tables = load_fixture("tiny_stages")
    env = GraDoomVecEnv(smap, lanes, device="cuda:0", render_mode="rgb_array")
    seeds = torch.arange(lanes, device="cuda:0")
    for shift in (0, 7):       # the second time over what the first left
        env.reset_device(torch.ones(lanes, dtype=torch.bool, device="cuda:0"), seeds + shift)
        rgb = torch.zeros((lanes, 240, 320, 3), dtype=torch.uint8, device="cuda:0")
        env._renderer.render(env._dynamics.lane_state(), rgb=rgb)
        frames = env.get_images()
        assert len(frames) == lanes and np.array_equal(np.stack(frames), rgb.cpu().numpy())
    env.close()


@pytest.mark.parametrize("where", ["class", "object"])
@pytest.mark.parametrize("lanes", [31, 32])   # fewer than two parts, two
def test_a_renderer_that_writes_rgb_frames_in_its_own_way_is_asked_for_them(lanes, where):
    from gradoom_amd.env import GraDoomVecEnv
    from gradoom_amd.renderer import HipRenderer

    class Marking(HipRenderer):
        def render_rgb_to_host(self, state, rgb):
            HipRenderer.render_rgb_to_host(self, state, rgb)
            torch.cuda.current_stream(self.device).synchronize()
            rgb[:, :8, :8] = 255

    class Refusing(HipRenderer):    # RGB frames never were a matter of render()
        def render(self, state, **out):
            assert "indexed" not in out
            HipRenderer.render(self, state, **out)

    _meta, _data, smap, _tables = load_fixture("tiny_stages")
    reset = torch.ones(lanes, dtype=torch.bool, device="cuda:0"), torch.arange(lanes, device="cuda:0")
    taken = []
    for kind in (HipRenderer, Marking, Refusing):
        renderer = (kind if where == "class" else HipRenderer)(smap, lanes, "cuda:0")
        if where == "object" and kind is not HipRenderer:
            name = "render_rgb_to_host" if kind is Marking else "render"
            setattr(renderer, name, getattr(kind, name).__get__(renderer))
        env = GraDoomVecEnv(smap, lanes, device="cuda:0", render_mode="rgb_array", renderer=renderer)
        env.reset_device(*reset)
        taken.append(np.stack(env.get_images()))
        env.close()
    plain, marked, refused = taken
    assert np.array_equal(plain, refused)
    plain[:, :8, :8] = 255
    assert np.array_equal(plain, marked)


@pytest.mark.parametrize("room", [1, 2, 64])   # frames that the pinned staging memory holds
def test_rgb_frames_are_arrays_of_their_own(monkeypatch, room):
    from gradoom_amd.env import GraDoomVecEnv

    monkeypatch.setattr(GraDoomVecEnv, "RGB_STAGING_BYTES", room * 240 * 320 * 3)
    _meta, _data, smap, _tables = load_fixture("tiny_stages")
    env = GraDoomVecEnv(smap, 5, device="cuda:0", render_mode="rgb_array")
    env.reset_device(torch.ones(5, dtype=torch.bool, device="cuda:0"), torch.arange(5, device="cuda:0"))
    rgb = torch.zeros((5, 240, 320, 3), dtype=torch.uint8, device="cuda:0")
    env._renderer.render(env._dynamics.lane_state(), rgb=rgb)
    expected = rgb.cpu().numpy()
    frames = env.get_images()
    assert len(frames) == 5 and all(np.array_equal(frame, expected[lane]) for lane, frame in enumerate(frames))
    assert np.array_equal(env.render_lane(3), expected[3])
    every = frames + env.get_images() + [env.render_lane(3)]
    for at, frame in enumerate(every):   # an array each, none of which keeps another's memory
        frame.fill(at)
    assert all(int(frame.min()) == int(frame.max()) == at and frame.nbytes == 240 * 320 * 3 for at, frame in enumerate(every))
    assert not any(np.shares_memory(frame, other) for at, frame in enumerate(every) for other in every[:at])
    held = every[1][5]
    frame = other = None
    every.clear()
    frames.clear()
    assert all(np.array_equal(frame, expected[lane]) for lane, frame in enumerate(env.get_images()))
    assert (held == 1).all()
    env.close()
