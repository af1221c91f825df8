"""Device-resident vector-env front end with the reference's render-path contract.

Mirrors the part of ``GraDoomVecEnv`` (``/root/reference/src/gradoom/env.py``) that
the render path serves:

* ``reset_device(mask, seeds) -> (observations, signals)``                      (``env.py:879-907``)
* ``step_device(actions) -> DeviceTransition``                                  (``env.py:851-877``)
* ``step_and_reset_device(actions, reset_seeds) -> DeviceAutoResetTransition``  (``env.py:909-942, 998``)
* ``render() / render_lane(i) / get_images()`` -> ``uint8 (240, 320, 3)``       (``env.py:1037-1064``)
* ``reset(seed=, options=) / step(actions)`` with ``obs_copy`` ownership         (``env.py:750-834, 678-688``)

with the same argument validation (``env.py:711-728``), the same ownership rules
(``observations`` is the renderer-owned ``frames`` stack returned by reference;
``final_*`` are fresh clones; the reset is skipped when no lane is done) and the
same error classes.  Gameplay (movement, combat, rewards) is NOT part of this
package: the lane state that the renderer draws comes from a ``LaneDynamics``
object.  ``PosePoolDynamics`` is a deterministic stand-in that teleports every
lane through a seeded pool of poses; a real engine would implement the same
three methods on top of its own state tensors.
"""

from __future__ import annotations

import collections
import ctypes as C
import dataclasses
import operator
import threading
import weakref
from collections.abc import Sequence

import numpy as np
import torch

from . import _abi, _lib, hostmath, synthmap
from .renderer import HipRenderer, LaneState

SIGNAL_COUNT = 27  # len(DEVICE_SIGNAL_NAMES), engine.py:509-539
INDEX_DTYPES = (torch.int8, torch.int16, torch.int32, torch.int64, torch.uint8)


@dataclasses.dataclass(frozen=True)
class DeviceTransition:  # env.py:181-190
    observations: torch.Tensor
    rewards: torch.Tensor
    terminated: torch.Tensor
    truncated: torch.Tensor
    signals: torch.Tensor
    info_histories: torch.Tensor


@dataclasses.dataclass(frozen=True)
class DeviceAutoResetTransition:  # env.py:193-205
    observations: torch.Tensor
    rewards: torch.Tensor
    terminated: torch.Tensor
    truncated: torch.Tensor
    signals: torch.Tensor
    info_histories: torch.Tensor
    final_observations: torch.Tensor
    final_signals: torch.Tensor
    final_info_histories: torch.Tensor


def _normalize_seed(seed, num_envs: int):  # env.py:101-113
    if seed is None:
        return [None] * num_envs
    if isinstance(seed, Sequence) and not isinstance(seed, (str, bytes, bytearray)):
        values = [None if value is None else int(value) for value in seed]
        if len(values) != num_envs:
            raise ValueError("seed sequence length must match num_envs")
        return values
    return [int(seed) + lane for lane in range(num_envs)]


def _stream(device) -> int:
    return torch.cuda.current_stream(device).cuda_stream


def _kernel_ready(tensor, dtype, count: int, device) -> bool:
    """Can a kernel of the library take this tensor as it is: ``count`` contiguous elements of ``dtype`` on ``device``?"""

    return isinstance(tensor, torch.Tensor) and tensor.dtype is dtype and tensor.shape == (count,) and tensor.device == device and tensor.is_contiguous()


def _own(method, function) -> bool:
    """Is this bound method the package's ``function``, and no other put in its place?"""

    return getattr(method, "__func__", None) is function


class _FramePool:
    """Host memory of RGB frames that their holders have let go of, for the next frames: at most ``limit`` frames of it.

    Every frame handed out is an array with memory of its own, which comes back when the array and every view of it are gone.
    The environments that hand frames out share one pool; what it keeps is freed with the last of them.
    """

    SHAPE = (240, 320, 3)

    class _Memory:
        __slots__ = ("array", "address", "interface")

        def __init__(self):
            self.array = np.empty(_FramePool.SHAPE, dtype=np.uint8)
            self.address, self.interface = self.array.ctypes.data, self.array.__array_interface__

    class _Lent:   # the base of a frame handed out: lives as long as the frame and its views
        __slots__ = ("_pool", "_memory", "__array_interface__")

        def __init__(self, pool, memory):
            self._pool, self._memory, self.__array_interface__ = pool, memory, memory.interface

        def __del__(self):
            if self._pool._users > 0:
                self._pool._free.append(self._memory)

    def __init__(self, limit: int):
        self._free = collections.deque(maxlen=limit)   # its operations are whole ones to other threads
        self._users = 0
        self._lock = threading.RLock()   # a user may be found gone while the thread holds it

    def join(self, user):
        """A call that ends ``user``'s part in the pool; made by itself when ``user`` is gone."""

        with self._lock:
            self._users += 1
        return weakref.finalize(user, self._leave)

    def _leave(self) -> None:
        with self._lock:
            self._users -= 1
            if self._users == 0:
                self._free.clear()

    def _memory(self) -> _Memory:
        try:
            return self._free.pop()
        except IndexError:
            return self._Memory()

    def copies_of(self, frames: np.ndarray) -> list[np.ndarray]:
        """Every frame of a contiguous ``uint8 [N, 240, 320, 3]``, each in memory of its own."""

        return self.filled_by(len(frames), lambda targets: _lib.check(_lib.library().gd_copy_pieces(frames.ctypes.data, targets, len(targets), 240 * 320 * 3)))

    def filled_by(self, count: int, fill) -> list[np.ndarray]:
        """``count`` frames in memory of their own, written by ``fill``, which is given their addresses."""

        memories = [self._memory() for _ in range(count)]
        fill((C.c_void_p * count)(*[memory.address for memory in memories]))
        return [np.asarray(self._Lent(self, memory)) for memory in memories]


RGB_STAGING_BYTES = 64 << 20   # of frames on their way to the host: pinned, an environment; let go of, all of them together
# Frames that are copied while others come.  get_images in us, all of them copied behind the last / 12 / 16 / 20 / 24 / 32 a part (two parts at least): 32 lanes
# 623 / 560 / 565, 48 lanes 747 / 689 / 672 / 648 / 673, 64 lanes 888 / 779 / 771 / 787 / 737 / 780, 128 lanes 1451 / 1175 / 1168 / 1175 / 1173 / 1204.
RGB_PART_FRAMES = 16
_FRAMES = _FramePool(RGB_STAGING_BYTES // (240 * 320 * 3))


class PosePoolDynamics:
    """Deterministic lane state source: lane ``i`` at time ``t`` shows pose ``(seed_i + t) mod pool``.

    On a ROCm device a step, a reset and the lane state are one kernel each (``gd_pose_step``, ``gd_pose_reset``,
    ``gd_pose_lanes``); elsewhere they are the Torch expressions below.
    """

    def __init__(self, smap, num_envs: int, device, *, pool: int = 64, sprites: int = 0, episode_timeout: int = 32, seed: int = 0):
        self.device = torch.device(device)
        self.num_envs = num_envs
        self.episode_timeout = int(episode_timeout)
        poses = synthmap.generate_poses_batch(smap, pool, seed, flash=True)
        to = lambda array, dtype: torch.as_tensor(np.ascontiguousarray(array)).to(device=self.device, dtype=dtype)  # noqa: E731
        self._pool = dict(
            x=to(poses.x, torch.float32), y=to(poses.y, torch.float32), view_z=to(poses.view_z, torch.float32),
            angle_bam=to(poses.angle_bam, torch.int64), pitch_bam=to(poses.pitch_bam, torch.int64),
            flash_light=to(poses.flash_light, torch.int64),
        )
        self._pool_size = pool
        self._sprites = None
        if sprites:
            spr = synthmap.generate_sprites_batch(smap, pool, sprites, seed)
            self._sprites = dict(
                sprite_x=to(spr.x, torch.float32), sprite_y=to(spr.y, torch.float32), sprite_z=to(spr.z, torch.float32),
                sprite_id=to(spr.sprite, torch.int32), sprite_alive=to(spr.alive.astype(np.uint8), torch.uint8),
                sprite_fullbright=to(spr.fullbright.astype(np.uint8), torch.uint8),
            )
        self.phase = torch.zeros(num_envs, dtype=torch.int64, device=self.device)
        self.episode_time = torch.zeros(num_envs, dtype=torch.int64, device=self.device)

    def _on_device(self, *tensors) -> bool:
        """Do the kernels take this call: the pool's own two counters and the call's tensors, each where and what it should be?"""

        if self.device.type != "cuda":
            return False
        device, count = self.phase.device, self.num_envs
        return (_kernel_ready(self.phase, torch.int64, count, device) and _kernel_ready(self.episode_time, torch.int64, count, device)
                and all(_kernel_ready(tensor, dtype, count, device) for tensor, dtype in tensors))

    def reset(self, mask: torch.Tensor, seeds: torch.Tensor) -> None:
        if self._on_device((mask, torch.bool), (seeds, torch.int64)):
            with torch.cuda.device(self.device):
                _lib.check(_lib.library().gd_pose_reset(self.phase.data_ptr(), self.episode_time.data_ptr(), mask.data_ptr(), seeds.data_ptr(), self.num_envs,
                                                        self._pool_size, _stream(self.device)))
            return
        self.phase.copy_(torch.where(mask, torch.remainder(seeds, self._pool_size), self.phase))
        self.episode_time.copy_(torch.where(mask, torch.zeros_like(self.episode_time), self.episode_time))

    def step(self, actions: torch.Tensor):
        if self._on_device((actions, torch.int64)):
            rewards = torch.empty(self.num_envs, dtype=torch.float32, device=self.device)
            terminated, truncated = torch.empty((2, self.num_envs), dtype=torch.bool, device=self.device).unbind(0)
            with torch.cuda.device(self.device):
                _lib.check(_lib.library().gd_pose_step(self.phase.data_ptr(), self.episode_time.data_ptr(), actions.data_ptr(), self.num_envs, self._pool_size,
                                                       self.episode_timeout, rewards.data_ptr(), terminated.data_ptr(), truncated.data_ptr(), _stream(self.device)))
            return rewards, terminated, truncated
        self.phase.copy_(torch.remainder(self.phase + 1 + actions, self._pool_size))
        self.episode_time.add_(1)
        rewards = torch.zeros(self.num_envs, dtype=torch.float32, device=self.device)
        terminated = torch.zeros(self.num_envs, dtype=torch.bool, device=self.device)
        truncated = self.episode_time >= self.episode_timeout
        return rewards, terminated, truncated

    def lane_state(self, rows: torch.Tensor | None = None) -> LaneState:
        """The lane state of every lane, or of the lanes that ``rows`` (indices of one dimension, on the device) names."""

        pool = self._pool
        taken = rows is None or (isinstance(rows, torch.Tensor) and rows.dim() == 1 and _kernel_ready(rows, torch.int64, rows.shape[0], self.phase.device))
        if taken and self._on_device() and all(value.is_contiguous() for value in pool.values()):
            return self._lane_state_kernel(rows)
        index = self.phase if rows is None else self.phase[rows]
        x, y = pool["x"][index], pool["y"][index]
        bam = pool["angle_bam"][index]
        fields = dict(
            x=x, y=y, angle=hostmath.angle_from_bam(bam), view_z=pool["view_z"][index],
            x_fixed=torch.round(x * 65536).to(torch.int64), y_fixed=torch.round(y * 65536).to(torch.int64),
            angle_bam=bam, pitch_bam=pool["pitch_bam"][index], flash_light=pool["flash_light"][index],
        )
        if self._sprites is not None:
            fields.update({name: value[index].contiguous() for name, value in self._sprites.items()})
        return LaneState(**{name: value.contiguous() for name, value in fields.items()})

    def _lane_state_kernel(self, rows) -> LaneState:
        count = self.num_envs if rows is None else int(rows.shape[0])
        device = self.device
        desc = _abi.PoseDesc()
        desc.lane_count, desc.pool_size, desc.phase, desc.phase_count = count, self._pool_size, self.phase.data_ptr(), self.num_envs
        if rows is not None:
            desc.rows = rows.data_ptr()
        pool = self._pool
        for name in ("x", "y", "view_z", "angle_bam", "pitch_bam", "flash_light"):
            setattr(desc, "pool_" + name, pool[name].data_ptr())
        fields = dict(zip(("x", "y", "angle", "view_z"), torch.empty((4, count), dtype=torch.float32, device=device).unbind(0)))
        fields.update(zip(("x_fixed", "y_fixed", "angle_bam", "pitch_bam", "flash_light"), torch.empty((5, count), dtype=torch.int64, device=device).unbind(0)))
        if self._sprites is not None:
            slots = int(self._sprites["sprite_x"].shape[1])
            desc.sprite_slots = slots
            for name, value in self._sprites.items():
                setattr(desc, "pool_" + name, value.data_ptr())
            fields.update(zip(("sprite_x", "sprite_y", "sprite_z"), torch.empty((3, count, slots), dtype=torch.float32, device=device).unbind(0)))
            fields["sprite_id"] = torch.empty((count, slots), dtype=torch.int32, device=device)
            fields.update(zip(("sprite_alive", "sprite_fullbright"), torch.empty((2, count, slots), dtype=torch.uint8, device=device).unbind(0)))
        for name, value in fields.items():
            setattr(desc, name, value.data_ptr())
        with torch.cuda.device(device):
            _lib.check(_lib.library().gd_pose_lanes(C.byref(desc), _stream(device)))
        return LaneState(**fields)


class GraDoomVecEnv:
    """Render-path subset of the reference's vector environment (device API only)."""

    frame_stack = 4

    def __init__(
        self,
        smap,
        num_envs: int,
        *,
        device="cuda:0",
        render_mode: str | None = None,
        obs_layout: str = "chw",
        obs_copy: str = "safe_view",
        dynamics=None,
        renderer=None,
        episode_timeout: int = 32,
        sprites: int = 0,
        action_count: int = 17,
    ):
        if num_envs <= 0:
            raise ValueError("num_envs must be positive")
        if obs_layout not in ("chw", "hwc"):
            raise ValueError("obs_layout must be 'chw' or 'hwc'")
        if obs_copy not in ("copy", "safe_view", "unsafe_view"):  # env.py:344-345
            raise ValueError("obs_copy must be copy, safe_view, or unsafe_view")
        if render_mode not in (None, "rgb_array"):
            raise ValueError("render_mode must be None or 'rgb_array'")
        self.num_envs = int(num_envs)
        self.device = torch.device(device)
        self._resident_device = self.device
        self.render_mode = render_mode
        self.obs_layout = obs_layout
        self.obs_copy = obs_copy
        self.observation_ownership = {"copy": "owned", "safe_view": "safe_view", "unsafe_view": "unsafe_view"}[obs_copy]  # env.py:377-382
        self.observation_buffer_depth = {"copy": None, "safe_view": 2, "unsafe_view": 1}[obs_copy]
        self.observation_renderer = "reference"
        self.closed = False
        self.action_count = int(action_count)   # len(action_table); 17 in the reference's pinned table (actions.py:33-51)
        if self.action_count <= 0:
            raise ValueError("action table must contain at least one action")
        self._renderer = renderer if renderer is not None else HipRenderer(smap, self.num_envs, self.device)
        self._dynamics = dynamics if dynamics is not None else PosePoolDynamics(
            smap, self.num_envs, self.device, sprites=sprites, episode_timeout=episode_timeout
        )
        n = self.num_envs
        # engine-owned buffers (engine.py:1927-1934)
        self.frames = torch.zeros((n, self.frame_stack, 84, 84), dtype=torch.uint8, device=self.device)
        self.signal_buffer = torch.zeros((n, SIGNAL_COUNT), dtype=torch.float32, device=self.device)
        self._info_history = torch.zeros((n, 0, self.frame_stack), dtype=torch.float32, device=self.device)
        self._initialized = torch.zeros(n, dtype=torch.bool, device=self.device)
        self.pending_reset = torch.ones(n, dtype=torch.bool, device=self.device)   # engine.py:1661
        self._latest_reset_seeds = torch.zeros(n, dtype=torch.int64, device=self.device)
        self._all_lanes = torch.ones(n, dtype=torch.uint8, device=self.device)
        # obs_copy="safe_view": two buffers handed out in turn, so that the observation of the step before stays
        # valid while this step's is written (env.py:459-472).  The renderer's observation kernel fills them.
        view_shape = (n, self.frame_stack, 84, 84) if obs_layout == "chw" else (n, 84, 84, self.frame_stack)
        self._view_shape = view_shape
        self._safe_obs_buffers = (
            tuple(torch.empty(view_shape, dtype=torch.uint8, device=self.device) for _ in range(2)) if obs_copy == "safe_view" else ()
        )
        self._safe_obs_index = 0
        # What the host wants to know of a step (gd_env_step, gd_env_check), in pinned memory: the kernels write it, a wait on the
        # stream makes it readable.
        self._native = self.device.type == "cuda"
        self._words = torch.zeros(16, dtype=torch.int32, pin_memory=True) if self._native else None
        self._words_read = self._words.numpy() if self._native else None
        self._done_rows = torch.zeros(n, dtype=torch.int64, device=self.device) if self._native else None
        self._drawn_mark = torch.cuda.Event() if self._native else None     # where a step's frames end
        self._rgb_staging = None        # pinned, at most RGB_STAGING_BYTES
        self._leave_frames = _FRAMES.join(self)
        self._seed_values = [None] * n
        self._done_listed = False       # did the last step's kernel list the lanes that ended?
        self._deferred_actions = None   # the one-element tuple step_async leaves for step_wait
        self._reset_rngs = [np.random.default_rng() for _ in range(n)]

    # ------------------------------------------------------------------ helpers
    def _require_device_tensor(self, value, name, *, shape, dtypes):  # env.py:711-728
        if not isinstance(value, torch.Tensor):
            raise TypeError(f"{name} must be a Torch tensor")
        if value.device != self._resident_device:
            raise TypeError(f"{name} must be on device {self._resident_device}")
        if value.shape != shape:
            raise ValueError(f"{name} must have shape {shape}")
        if value.dtype not in dtypes:
            expected = ", ".join(str(dtype) for dtype in dtypes)
            raise TypeError(f"{name} must have dtype {expected}")
        return value

    def _device_observations(self, observations: torch.Tensor) -> torch.Tensor:  # env.py:690-691
        return observations.permute(0, 2, 3, 1) if self.obs_layout == "hwc" else observations

    def _bookkeeping_ready(self) -> bool:
        """Are the tensors of a step's bookkeeping what the kernels take?  (A dynamics object may keep its clock in another type.)"""

        return self._native and _kernel_ready(self._dynamics.episode_time, torch.int64, self.num_envs, self.frames.device)

    def _wait(self) -> None:
        torch.cuda.current_stream(self.device).synchronize()

    def _update_signals(self) -> None:
        self.signal_buffer[:, 17].copy_(self._dynamics.episode_time)  # episode_time, engine.py:15469
        self.signal_buffer[:, 20].copy_(self.pending_reset)           # engine.py:15472

    # ------------------------------------------------------------------ device API
    def reset_device(self, mask: torch.Tensor, seeds: torch.Tensor):
        return self._reset(mask, seeds, None)

    def _reset(self, mask: torch.Tensor, seeds: torch.Tensor, view):
        if self.closed:
            raise RuntimeError("cannot reset a closed environment")
        device_mask = self._require_device_tensor(mask, "mask", shape=(self.num_envs,), dtypes=(torch.bool,))
        device_seeds = self._require_device_tensor(seeds, "seeds", shape=(self.num_envs,), dtypes=INDEX_DTYPES).to(torch.int64)
        self._dynamics.reset(device_mask, device_seeds)
        # engine.reset renders every lane and fills the stack of the masked ones with four copies
        # (engine.py:2443-2450); unmasked lanes keep their stack, which the fused epilogue does by
        # writing only under the mask.
        self._renderer.render(self._dynamics.lane_state(), frames=self.frames, reset_mask=device_mask, obs=None, stack_only_masked=True,
                              final_frames=view, final_layout=self.obs_layout)
        self._after_reset(device_mask, device_seeds)
        return self._device_observations(self.frames), self.signal_buffer

    def _after_reset(self, device_mask: torch.Tensor, device_seeds: torch.Tensor) -> None:
        if self._bookkeeping_ready() and device_mask.is_contiguous() and device_seeds.is_contiguous():
            with torch.cuda.device(self.device):
                _lib.check(_lib.library().gd_env_reset(device_mask.data_ptr(), device_seeds.data_ptr(), self._dynamics.episode_time.data_ptr(), self.num_envs,
                                                       self._latest_reset_seeds.data_ptr(), self._initialized.data_ptr(), self.pending_reset.data_ptr(),
                                                       self.signal_buffer.data_ptr(), _stream(self.device)))
            return
        self._latest_reset_seeds.copy_(torch.where(device_mask, device_seeds, self._latest_reset_seeds))
        self._initialized |= device_mask
        self.pending_reset.masked_fill_(device_mask, False)   # engine.py:2409
        self._update_signals()

    def _resets_alone(self) -> bool:
        """May the lanes that end be rendered alone, around ``reset_device`` and the renderer's own stack update?

        Only where both are this package's: an environment that overrides ``reset_device`` has it called, and another renderer
        is asked for the frames of all lanes with a reset mask, as its interface has it.
        """

        return _own(self.reset_device, GraDoomVecEnv.reset_device) and _own(getattr(self._renderer, "render", None), HipRenderer.render)

    def _lane_rows(self, rows: torch.Tensor) -> LaneState:
        """The lane state of some lanes.  A dynamics object owes ``lane_state()`` and no more; the pool's own also takes the lanes."""

        lane_state = self._dynamics.lane_state
        if getattr(lane_state, "__func__", None) is PosePoolDynamics.lane_state:
            return lane_state(rows)
        return lane_state().select(rows)

    def _reset_rows(self, device_mask: torch.Tensor, seeds: torch.Tensor, count: int):
        """``_reset`` of the ``count`` lanes that ``_done_rows`` lists: only they are rendered, four copies each into their stacks."""

        device_seeds = self._require_device_tensor(seeds, "seeds", shape=(self.num_envs,), dtypes=INDEX_DTYPES).to(torch.int64).contiguous()
        self._dynamics.reset(device_mask, device_seeds)
        rows = self._done_rows[:count]
        state = self._lane_rows(rows)
        obs = torch.empty((count, 84, 84), dtype=torch.uint8, device=self.device)
        self._renderer.render(state, obs=obs)
        with torch.cuda.device(self.device):
            _lib.check(_lib.library().gd_fill_stacks(obs.data_ptr(), rows.data_ptr(), count, self.frames.data_ptr(), _stream(self.device)))
        self._after_reset(device_mask, device_seeds)
        return self._device_observations(self.frames), self.signal_buffer

    def step_device(self, actions: torch.Tensor) -> DeviceTransition:
        return self._step(actions, None)

    def _after_step(self, terminated, truncated, list_done: bool) -> bool:
        """The bookkeeping of a step in one kernel; false where its tensors are not what the kernel takes."""

        device, count = self.frames.device, self.num_envs
        if not (self._bookkeeping_ready() and _kernel_ready(terminated, torch.bool, count, device) and _kernel_ready(truncated, torch.bool, count, device)):
            return False
        with torch.cuda.device(self.device):
            _lib.check(_lib.library().gd_env_step(terminated.data_ptr(), truncated.data_ptr(), self._dynamics.episode_time.data_ptr(), count,
                                                  self.pending_reset.data_ptr(), self.signal_buffer.data_ptr(), self._done_rows.data_ptr() if list_done else None,
                                                  self._words.data_ptr() if list_done else None, _stream(self.device)))
        return True

    def _step(self, actions: torch.Tensor, final_frames, final_layout: str = "chw", list_done: bool = False) -> DeviceTransition:
        if self.closed:
            raise RuntimeError("cannot step a closed environment")
        indices = self._require_device_tensor(actions, "actions", shape=(self.num_envs,), dtypes=INDEX_DTYPES).to(torch.int64)
        rewards, terminated, truncated = self._dynamics.step(indices)
        self._done_listed = self._after_step(terminated, truncated, list_done)
        if not self._done_listed:
            self.pending_reset.copy_(terminated | truncated)      # engine.py:9542
        lanes, marks = self._dynamics.lane_state(), self._done_listed and list_done
        if marks and self._resets_alone():
            self._renderer.mark_status()
        self._renderer.render(lanes, frames=self.frames, final_frames=final_frames, final_layout=final_layout)
        if marks:
            self._drawn_mark.record(torch.cuda.current_stream(self.device))
        if not self._done_listed:
            self._update_signals()
        return DeviceTransition(
            observations=self._device_observations(self.frames), rewards=rewards, terminated=terminated, truncated=truncated,
            signals=self.signal_buffer, info_histories=self._info_history,
        )

    def step_and_reset_device(self, actions: torch.Tensor, reset_seeds: torch.Tensor) -> DeviceAutoResetTransition:
        """``step_device``, then ``reset_device`` of the lanes that ended (env.py:908-940).

        Raises ``RuntimeError`` where the renderer truncated one of the step's frames: the step has been taken, no lane has been reset
        (``pending_reset`` says which have ended) and the seeds have not been looked at.
        """

        # the final-observation clone (env.py:915) is written by the observation kernel of the step
        final_frames = torch.empty_like(self.frames)
        transition = self._step(actions, final_frames, list_done=True)
        final_observations = self._device_observations(final_frames)
        final_signals = transition.signals.clone()
        final_info_histories = transition.info_histories.clone()
        listed = self._done_listed
        alone = listed and self._resets_alone()
        if alone:    # how many lanes ended, and whether a frame was truncated, is known while the step's frames are still being put together
            self._renderer.wait_status()
            done_count = int(self._words_read[0])
            alone = 0 < done_count <= 65535
        elif listed:   # one wait on the stream
            self._wait()
            done_count = int(self._words_read[0])
        else:
            done = transition.terminated | transition.truncated
            done_count = int(torch.count_nonzero(done))  # env.py:919: one host sync for the reference renderer
        if alone:    # refused, a step leaves the lanes that ended as they are: none of the reset has begun
            self._refuse_truncated(self._renderer.status_seen())
            # the reset is queued behind the step's frames: the device goes from one to the other without the host
            observations, signals = self._reset_rows(self.pending_reset.clone(), reset_seeds, done_count)
            self._drawn_mark.synchronize()
        else:
            self.check_renderer_status()
        if not done_count:
            return DeviceAutoResetTransition(
                transition.observations, transition.rewards, transition.terminated, transition.truncated,
                transition.signals, transition.info_histories, final_observations, final_signals, final_info_histories,
            )
        if not alone:
            done = transition.terminated | transition.truncated
            observations, signals = self.reset_device(done, reset_seeds)
        return DeviceAutoResetTransition(
            observations, transition.rewards, transition.terminated, transition.truncated, signals, self._info_history,
            final_observations, final_signals, final_info_histories,
        )

    def device_signals(self) -> torch.Tensor:
        return self.signal_buffer

    def check_renderer_status(self) -> None:
        """Raise if the renderer had to drop a linedef from a column's candidate list.

        A column keeps 64 linedefs in its own slots and up to 256 in the spill pool, which holds one column in 32 of a large
        batch (every column of up to eight lanes).

        Such a frame may differ from the reference's, which has no such bound, so it must not pass for a good one.
        Waits for the current stream (called where the environment has waited for it already): what other streams run goes on.
        """
        status = getattr(self._renderer, "status_seen", None)
        if status is not None and self._native:
            self._wait()
        elif status is None:
            status = getattr(self._renderer, "status", None)
        self._refuse_truncated(status() if status is not None else 0)

    def _refuse_truncated(self, flags: int) -> None:
        if flags & 1:
            raise RuntimeError(
                "the renderer truncated a screen column's candidate list (more than 256 linedefs overlap one column of one "
                "lane's view, or more columns than the spill pool holds see more than 64): frames of this environment are "
                "not trustworthy on this map"
            )
        if flags & 2:
            raise RuntimeError(
                "the renderer truncated a screen column's list of drawsegs (a column crossed more than 255 portals): frames of "
                "this environment are not trustworthy on this map"
            )

    # ------------------------------------------------------------------ host-facing API (env.py:750-834)
    def _view_target(self):
        """The tensor this call's observation copy goes to, or None for ``unsafe_view`` (env.py:678-688)."""
        if self.obs_copy == "copy":
            return torch.empty(self._view_shape, dtype=torch.uint8, device=self.device)
        if self.obs_copy == "safe_view":
            buffer = self._safe_obs_buffers[self._safe_obs_index]
            self._safe_obs_index = (self._safe_obs_index + 1) % len(self._safe_obs_buffers)
            return buffer
        return None

    def seed(self, seed=None):
        self._seed_values = _normalize_seed(seed, self.num_envs)
        return list(self._seed_values)

    def reset(self, *, seed=None, options=None):
        if self.closed:
            raise RuntimeError("cannot reset a closed environment")
        reset_options = dict(options or {})
        raw_mask = reset_options.pop("reset_mask", None)
        if raw_mask is None:
            mask = torch.ones(self.num_envs, device=self.device, dtype=torch.bool)
        else:
            mask = self._require_device_tensor(raw_mask, "options['reset_mask']", shape=(self.num_envs,), dtypes=(torch.bool,))
        if not bool(torch.any(mask)):
            raise ValueError("options['reset_mask'] must select at least one lane")
        if reset_options:
            raise ValueError(f"unsupported reset options: {sorted(reset_options)}")
        seed_values = _normalize_seed(seed, self.num_envs) if seed is not None else self._seed_values
        game_seeds = [0] * self.num_envs
        for lane in torch.nonzero(mask, as_tuple=False).flatten().to("cpu").tolist():
            if seed_values[lane] is not None:
                self._reset_rngs[lane] = np.random.default_rng(seed_values[lane])
            game_seeds[lane] = int(self._reset_rngs[lane].integers(0, np.iinfo(np.uint32).max + 1, dtype=np.uint32))
        self._seed_values = [None] * self.num_envs
        seeds = torch.tensor(game_seeds, device=self.device, dtype=torch.int64)
        view = self._view_target()
        observations, _ = self._reset(mask, seeds, view)
        return (observations if view is None else view), {}

    def _check_step(self, actions):
        """(some lane was never reset, some lane has ended, some action is out of range); the last None where that was not looked at."""

        if not self._native:
            return not bool(torch.all(self._initialized)), bool(torch.any(self.pending_reset)), None
        looked_at = _kernel_ready(actions, torch.int64, self.num_envs, self.frames.device)
        with torch.cuda.device(self.device):
            _lib.check(_lib.library().gd_env_check(self._initialized.data_ptr(), self.pending_reset.data_ptr(), actions.data_ptr() if looked_at else None,
                                                   self.num_envs, self.action_count, self._words.data_ptr() + 4, _stream(self.device)))
        self._wait()
        flags = int(self._words_read[1])
        return bool(flags & 1), bool(flags & 2), bool(flags & 4) if looked_at else None

    def step(self, actions: torch.Tensor):
        if self.closed:
            raise RuntimeError("cannot step a closed environment")
        uninitialized, pending, outside = self._check_step(actions)
        if uninitialized:
            raise RuntimeError("all lanes must be reset before the first step")
        if pending:   # env.py:819-821
            lanes = torch.nonzero(self.pending_reset).flatten().to("cpu").tolist()
            raise RuntimeError(f"terminal lanes must be reset before step: {lanes}")
        # every argument is checked before the observation buffer is taken: a refused call must not advance the
        # safe_view rotation, or the next step would write into the buffer the caller still holds (env.py:459-472)
        indices = self._require_device_tensor(actions, "actions", shape=(self.num_envs,), dtypes=INDEX_DTYPES).to(torch.int64)
        if outside if outside is not None else bool(torch.any((indices < 0) | (indices >= self.action_count))):   # env.py:828-829
            raise ValueError("actions fall outside the declared action space")
        view = self._view_target()
        transition = self._step(indices, view, self.obs_layout)
        observations = transition.observations if view is None else view
        return observations, transition.rewards, transition.terminated, transition.truncated, {}

    def step_async(self, actions: torch.Tensor) -> None:  # env.py:839-842
        """Hand in the actions of a step that ``step_wait`` will run; nothing is checked or rendered yet."""
        if self._deferred_actions is not None:
            raise RuntimeError("an asynchronous step is already pending")
        self._deferred_actions = (actions,)

    def step_wait(self):  # env.py:844-849
        if self._deferred_actions is None:
            raise RuntimeError("no asynchronous step is pending")
        (actions,), self._deferred_actions = self._deferred_actions, None
        return self.step(actions)

    # ------------------------------------------------------------------ RGB frames
    RGB_STAGING_BYTES = RGB_STAGING_BYTES

    def _rgb_frames(self, lane: int | None = None) -> list[np.ndarray]:
        """RGB frames of all lanes, or of one, each a host array of its own (a caller that keeps one keeps no other alive)."""

        state = self._dynamics.lane_state()
        if lane is not None and self.num_envs > 1:   # one lane's frame: only that lane is rendered
            state = state.select(slice(lane, lane + 1))
        count = int(state.x.shape[0])
        render_to_host = getattr(self._renderer, "render_rgb_to_host", None)
        if not self._native or render_to_host is None:
            rgb = torch.empty((count, 240, 320, 3), dtype=torch.uint8, device=self.device)
            self._renderer.render(state, rgb=rgb)
            return [frame.copy() for frame in rgb.detach().to("cpu").numpy()]
        # The expansion writes the frames into pinned host memory, over PCIe, as it makes them: no second copy of them on the device
        # and no staging by the runtime.  Each frame then goes to memory of its own, which was touched before where it can be (hence the
        # pool: fresh pages cost several times the copy).
        frame_bytes = 240 * 320 * 3
        room = max(1, min(count, self.RGB_STAGING_BYTES // frame_bytes))
        if self._rgb_staging is None or self._rgb_staging.shape[0] < room:
            self._rgb_staging = torch.empty((room, 240, 320, 3), dtype=torch.uint8, pin_memory=True)
        # By parts only where `render_rgb_to_host`, which is asked otherwise, and `render` are this package's.
        by_parts = state.screen_blend is None and _own(render_to_host, HipRenderer.render_rgb_to_host) and _own(getattr(self._renderer, "render", None), HipRenderer.render)
        frames = []
        for base in range(0, count, room):
            part = min(room, count - base)
            staging = self._rgb_staging[:part]
            lanes = state if part == count else state.select(slice(base, base + part))
            if by_parts and part >= 2 * RGB_PART_FRAMES:
                frames += self._rgb_in_parts(lanes, staging)
            else:
                render_to_host(lanes, staging)
                self._wait()
                frames += _FRAMES.copies_of(staging.numpy())
        return frames

    def _rgb_in_parts(self, lanes, staging: torch.Tensor) -> list[np.ndarray]:
        """The frames of many lanes: while some are on their way over PCIe, those that have come are copied to memory of their own."""

        indexed = torch.empty(tuple(staging.shape[:3]), dtype=torch.uint8, device=self.device)
        self._renderer.render(lanes, indexed=indexed)
        return _FRAMES.filled_by(len(staging), lambda targets: self._renderer.expand_rgb_to_pieces(indexed, staging, RGB_PART_FRAMES, targets))

    def render_lane(self, lane: int):  # env.py:1037-1053
        if self.closed:
            raise RuntimeError("cannot render a closed environment")
        if isinstance(lane, (bool, np.bool_)):
            raise TypeError("lane must be an integer")
        lane_index = operator.index(lane)
        if not 0 <= lane_index < self.num_envs:
            raise IndexError(f"lane must be in [0, {self.num_envs - 1}]")
        if self.render_mode != "rgb_array":
            return None
        frame = self._rgb_frames(lane_index)[0]
        self.check_renderer_status()
        return frame

    def render(self):
        return self.render_lane(0)

    def get_images(self):  # env.py:1058-1064
        if self.closed:
            raise RuntimeError("cannot render a closed environment")
        if self.render_mode != "rgb_array":
            return [None for _ in range(self.num_envs)]
        frames = self._rgb_frames()
        self.check_renderer_status()
        return frames

    def close(self) -> None:
        if not self.closed:
            self.closed = True
            self._leave_frames()
            try:
                if self._native:
                    torch.cuda.synchronize(self.device)   # frames may have been drawn on any stream
                self.check_renderer_status()
            finally:
                self._close_renderer()

    def _close_renderer(self) -> None:
        close = getattr(self._renderer, "close", None)
        if close is not None:
            close()
