// What a vector environment does around its frames, one kernel each: the lane state of a pose pool, a step and a reset of that pool,
// the checks and the bookkeeping of a step.  As Torch operators these were some forty launches a step, five to ten microseconds of
// host time each and, on small batches, the larger part of the step; what the host has to know (is a lane done, is an action out of
// range) is written to pinned host memory, so that one wait on the stream answers all of it.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <exception>
#include <string>
#include <thread>
#include <vector>

#include "../../include/gradoom_amd.h"
#include "gd_internal.h"

namespace {

typedef long long i64;

// torch.remainder: the sign of the divisor (positive here)
__device__ __forceinline__ i64 floor_mod(i64 v, i64 n) { const i64 r = v % n; return r < 0 ? r + n : r; }

#define POSE_THREADS 128
// One work-group per lane: its pose by the first threads, its billboards by all of them.
__global__ void __launch_bounds__(POSE_THREADS) pose_lanes_kernel(gd_pose_desc d) {
    const int lane = blockIdx.x;
    // a negative index counts from the end; one beyond either end is the one there
    auto inside = [](i64 at, i64 count) { at = at < 0 ? at + count : at; return at < 0 ? 0 : (at >= count ? count - 1 : at); };
    const i64 pose = inside(d.phase[d.rows ? inside(d.rows[lane], d.phase_count) : lane], d.pool_size);
    if (threadIdx.x == 0) {
        const float BAM_TO_RADIANS = (float)(2.0 * 3.14159265358979323846 / 4294967296.0);   // engine.py:10651
        const float x = d.pool_x[pose], y = d.pool_y[pose];
        const i64 bam = d.pool_angle_bam[pose];
        d.x[lane] = x; d.y[lane] = y; d.view_z[lane] = d.pool_view_z[pose];
        d.angle[lane] = (float)bam * BAM_TO_RADIANS;
        d.x_fixed[lane] = (i64)rintf(x * 65536.0f); d.y_fixed[lane] = (i64)rintf(y * 65536.0f);
        d.angle_bam[lane] = bam; d.pitch_bam[lane] = d.pool_pitch_bam[pose]; d.flash_light[lane] = d.pool_flash_light[pose];
    }
    for (int k = threadIdx.x; k < d.sprite_slots; k += POSE_THREADS) {
        const size_t from = (size_t)pose * d.sprite_slots + k, to = (size_t)lane * d.sprite_slots + k;
        d.sprite_x[to] = d.pool_sprite_x[from]; d.sprite_y[to] = d.pool_sprite_y[from]; d.sprite_z[to] = d.pool_sprite_z[from];
        d.sprite_id[to] = d.pool_sprite_id[from];
        d.sprite_alive[to] = d.pool_sprite_alive[from]; d.sprite_fullbright[to] = d.pool_sprite_fullbright[from];
    }
}

__global__ void __launch_bounds__(256) pose_step_kernel(int64_t *phase, int64_t *episode_time, const int64_t *actions, int count, i64 pool, i64 timeout,
                                                        float *rewards, uint8_t *terminated, uint8_t *truncated) {
    const int lane = blockIdx.x * blockDim.x + threadIdx.x;
    if (lane >= count) return;
    const i64 time = (i64)episode_time[lane] + 1;
    phase[lane] = floor_mod((i64)((uint64_t)phase[lane] + 1u + (uint64_t)actions[lane]), pool);
    episode_time[lane] = time;
    rewards[lane] = 0.0f; terminated[lane] = 0; truncated[lane] = time >= timeout ? 1 : 0;
}

__global__ void __launch_bounds__(256) pose_reset_kernel(int64_t *phase, int64_t *episode_time, const uint8_t *mask, const int64_t *seeds, int count, i64 pool) {
    const int lane = blockIdx.x * blockDim.x + threadIdx.x;
    if (lane >= count || !mask[lane]) return;
    phase[lane] = floor_mod(seeds[lane], pool);
    episode_time[lane] = 0;
}

#define SIGNAL_COUNT 27        // engine.py:509-539
#define SIGNAL_TIME 17         // episode_time, engine.py:15469
#define SIGNAL_PENDING 20      // pending_reset, engine.py:15472
#define ENV_THREADS 1024

// One work-group, a thread a lane at a time: the lanes that end are listed in lane order, so their places come from a running
// count over the work-group's wavefronts.
__global__ void __launch_bounds__(ENV_THREADS) env_step_kernel(const uint8_t *terminated, const uint8_t *truncated, const int64_t *episode_time, int count,
                                                               uint8_t *pending, float *signals, int64_t *done_rows, int32_t *done_count) {
    __shared__ int wave_count[ENV_THREADS / 64];
    const int wave = threadIdx.x >> 6, lane_id = threadIdx.x & 63;
    int listed = 0;
    for (int base = 0; base < count; base += ENV_THREADS) {
        const int lane = base + (int)threadIdx.x;
        const bool done = lane < count && (terminated[lane] || truncated[lane]);
        if (lane < count) {
            pending[lane] = done ? 1 : 0;
            signals[(size_t)lane * SIGNAL_COUNT + SIGNAL_TIME] = (float)(i64)episode_time[lane];
            signals[(size_t)lane * SIGNAL_COUNT + SIGNAL_PENDING] = done ? 1.0f : 0.0f;
        }
        if (!done_rows) continue;
        const unsigned long long ended = __ballot(done);
        if (lane_id == 0) wave_count[wave] = __popcll(ended);
        __syncthreads();
        int before = listed, total = 0;
        for (int w = 0; w < ENV_THREADS / 64; ++w) { before += w < wave ? wave_count[w] : 0; total += wave_count[w]; }
        if (done) done_rows[before + __popcll(ended & ((1ULL << lane_id) - 1))] = lane;
        listed += total;
        __syncthreads();
    }
    if (done_count && threadIdx.x == 0) *done_count = listed;
}

__global__ void __launch_bounds__(256) env_reset_kernel(const uint8_t *mask, const int64_t *seeds, const int64_t *episode_time, int count, int64_t *latest_seeds,
                                                        uint8_t *initialized, uint8_t *pending, float *signals) {
    const int lane = blockIdx.x * blockDim.x + threadIdx.x;
    if (lane >= count) return;
    const bool resets = mask[lane] != 0;
    if (resets) { latest_seeds[lane] = seeds[lane]; initialized[lane] = 1; pending[lane] = 0; }
    signals[(size_t)lane * SIGNAL_COUNT + SIGNAL_TIME] = (float)(i64)episode_time[lane];
    signals[(size_t)lane * SIGNAL_COUNT + SIGNAL_PENDING] = pending[lane] ? 1.0f : 0.0f;
}

__global__ void __launch_bounds__(ENV_THREADS) env_check_kernel(const uint8_t *initialized, const uint8_t *pending, const int64_t *actions, int count,
                                                                int action_count, int32_t *flags) {
    int found = 0;
    for (int lane = threadIdx.x; lane < count; lane += ENV_THREADS) {
        found |= (initialized[lane] ? 0 : 1) | (pending[lane] ? 2 : 0);
        if (actions) found |= actions[lane] < 0 || actions[lane] >= action_count ? 4 : 0;
    }
    const int uninitialized = __syncthreads_or(found & 1), ended = __syncthreads_or(found & 2), outside = __syncthreads_or(found & 4);
    if (threadIdx.x == 0) *flags = (uninitialized ? 1 : 0) | (ended ? 2 : 0) | (outside ? 4 : 0);
}

// Four copies of an observation each: the stacks of the lanes that `rows` names (engine.py:2443-2450).
__global__ void __launch_bounds__(256) fill_stacks_kernel(const unsigned int *obs, const int64_t *rows, unsigned int *frames) {
    const size_t words = (size_t)GD_OBS_SIZE * GD_OBS_SIZE / 4;
    const size_t lane = (size_t)rows[blockIdx.y];
    const size_t word = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (word >= words) return;
    const unsigned int v = obs[(size_t)blockIdx.y * words + word];
    for (int k = 0; k < GD_FRAME_STACK; ++k) frames[(lane * GD_FRAME_STACK + k) * words + word] = v;
}

dim3 lanes_of(int count) { return dim3((unsigned)((count + 255) / 256)); }

}  // namespace

extern "C" {

int gd_pose_lanes(const gd_pose_desc *d, void *stream) {
    if (!d) return gd_fail(GD_E_ARG, "null argument");
    GD_SIZE_CHECK(d, gd_pose_desc);
    if (d->lane_count < 0 || d->sprite_slots < 0 || d->pool_size <= 0 || d->phase_count <= 0 || (!d->rows && d->lane_count > d->phase_count))
        return gd_fail(GD_E_ARG, "gd_pose_desc holds a count out of range");
    if (d->lane_count == 0) return GD_OK;
    const void *const needed[] = {d->phase, d->pool_x, d->pool_y, d->pool_view_z, d->pool_angle_bam, d->pool_pitch_bam, d->pool_flash_light,
                                  d->x, d->y, d->angle, d->view_z, d->x_fixed, d->y_fixed, d->angle_bam, d->pitch_bam, d->flash_light};
    for (const void *p : needed) if (!p) return gd_fail(GD_E_ARG, "null tensor in gd_pose_desc");
    const void *const sprites[] = {d->pool_sprite_x, d->pool_sprite_y, d->pool_sprite_z, d->pool_sprite_id, d->pool_sprite_alive, d->pool_sprite_fullbright,
                                   d->sprite_x, d->sprite_y, d->sprite_z, d->sprite_id, d->sprite_alive, d->sprite_fullbright};
    for (const void *p : sprites) if (!p && d->sprite_slots > 0) return gd_fail(GD_E_ARG, "null billboard tensor in gd_pose_desc");
    hipLaunchKernelGGL(pose_lanes_kernel, dim3((unsigned)d->lane_count), dim3(POSE_THREADS), 0, static_cast<hipStream_t>(stream), *d);
    GD_HIP_TRY(hipGetLastError());
    return GD_OK;
}

int gd_pose_step(int64_t *phase, int64_t *episode_time, const int64_t *actions, int32_t lane_count, int64_t pool_size, int64_t episode_timeout,
                 float *rewards, uint8_t *terminated, uint8_t *truncated, void *stream) {
    if (lane_count < 0 || pool_size <= 0) return gd_fail(GD_E_ARG, "count out of range");
    if (lane_count == 0) return GD_OK;
    if (!phase || !episode_time || !actions || !rewards || !terminated || !truncated) return gd_fail(GD_E_ARG, "null argument");
    hipLaunchKernelGGL(pose_step_kernel, lanes_of(lane_count), dim3(256), 0, static_cast<hipStream_t>(stream), phase, episode_time, actions, lane_count, pool_size,
                       episode_timeout, rewards, terminated, truncated);
    GD_HIP_TRY(hipGetLastError());
    return GD_OK;
}

int gd_pose_reset(int64_t *phase, int64_t *episode_time, const uint8_t *mask, const int64_t *seeds, int32_t lane_count, int64_t pool_size, void *stream) {
    if (lane_count < 0 || pool_size <= 0) return gd_fail(GD_E_ARG, "count out of range");
    if (lane_count == 0) return GD_OK;
    if (!phase || !episode_time || !mask || !seeds) return gd_fail(GD_E_ARG, "null argument");
    hipLaunchKernelGGL(pose_reset_kernel, lanes_of(lane_count), dim3(256), 0, static_cast<hipStream_t>(stream), phase, episode_time, mask, seeds, lane_count, pool_size);
    GD_HIP_TRY(hipGetLastError());
    return GD_OK;
}

int gd_env_step(const uint8_t *terminated, const uint8_t *truncated, const int64_t *episode_time, int32_t lane_count, uint8_t *pending, float *signals,
                int64_t *done_rows, int32_t *done_count, void *stream) {
    if (lane_count <= 0) return gd_fail(GD_E_ARG, "count out of range");
    if (!terminated || !truncated || !episode_time || !pending || !signals) return gd_fail(GD_E_ARG, "null argument");
    hipLaunchKernelGGL(env_step_kernel, dim3(1), dim3(ENV_THREADS), 0, static_cast<hipStream_t>(stream), terminated, truncated, episode_time, lane_count, pending,
                       signals, done_rows, done_count);
    GD_HIP_TRY(hipGetLastError());
    return GD_OK;
}

int gd_env_reset(const uint8_t *mask, const int64_t *seeds, const int64_t *episode_time, int32_t lane_count, int64_t *latest_seeds, uint8_t *initialized,
                 uint8_t *pending, float *signals, void *stream) {
    if (lane_count <= 0) return gd_fail(GD_E_ARG, "count out of range");
    if (!mask || !seeds || !episode_time || !latest_seeds || !initialized || !pending || !signals) return gd_fail(GD_E_ARG, "null argument");
    hipLaunchKernelGGL(env_reset_kernel, lanes_of(lane_count), dim3(256), 0, static_cast<hipStream_t>(stream), mask, seeds, episode_time, lane_count, latest_seeds,
                       initialized, pending, signals);
    GD_HIP_TRY(hipGetLastError());
    return GD_OK;
}

int gd_env_check(const uint8_t *initialized, const uint8_t *pending, const int64_t *actions, int32_t lane_count, int32_t action_count, int32_t *flags, void *stream) {
    if (lane_count <= 0) return gd_fail(GD_E_ARG, "count out of range");
    if (!initialized || !pending || !flags) return gd_fail(GD_E_ARG, "null argument");
    hipLaunchKernelGGL(env_check_kernel, dim3(1), dim3(ENV_THREADS), 0, static_cast<hipStream_t>(stream), initialized, pending, actions, lane_count, action_count, flags);
    GD_HIP_TRY(hipGetLastError());
    return GD_OK;
}

int gd_fill_stacks(const uint8_t *obs, const int64_t *rows, int32_t count, uint8_t *frames, void *stream) {
    if (count < 0 || count > 65535) return gd_fail(GD_E_ARG, "count out of range");
    if (count == 0) return GD_OK;
    if (!obs || !rows || !frames) return gd_fail(GD_E_ARG, "null argument");
    if ((reinterpret_cast<size_t>(obs) | reinterpret_cast<size_t>(frames)) & 3) return gd_fail(GD_E_ARG, "obs and frames must be word aligned");
    const int words = GD_OBS_SIZE * GD_OBS_SIZE / 4;
    hipLaunchKernelGGL(fill_stacks_kernel, dim3((unsigned)((words + 255) / 256), (unsigned)count), dim3(256), 0, static_cast<hipStream_t>(stream),
                       reinterpret_cast<const unsigned int *>(obs), rows, reinterpret_cast<unsigned int *>(frames));
    GD_HIP_TRY(hipGetLastError());
    return GD_OK;
}

// Most of such a copy is waiting for memory the device has just written, or for fresh pages: the caller's thread and up to three more take
// every fourth piece.  48 frames of 230,400 bytes: 0.29 ms by one thread, 0.18 by four, 0.23 by eight.
int gd_copy_pieces(const void *source, void *const *targets, int32_t count, int64_t bytes) {
    if (count < 0 || bytes < 0) return gd_fail(GD_E_ARG, "count out of range");
    if (count == 0 || bytes == 0) return GD_OK;
    if (!source || !targets) return gd_fail(GD_E_ARG, "null argument");
    for (int32_t k = 0; k < count; ++k) if (!targets[k]) return gd_fail(GD_E_ARG, "null target");
    constexpr int THREADS = 4;
    auto copy = [=](int first) { for (int64_t k = first; k < count; k += THREADS) std::memcpy(targets[k], static_cast<const char *>(source) + k * bytes, (size_t)bytes); };
    std::thread helpers[THREADS - 1];
    for (int t = 1; t < THREADS; ++t) {
        if (count <= t || bytes * count < (1 << 20)) { copy(t); continue; }      // too little to be worth a thread
        try { helpers[t - 1] = std::thread(copy, t); } catch (const std::exception &) { copy(t); }   // no thread to be had
    }
    copy(0);
    for (std::thread &helper : helpers) if (helper.joinable()) helper.join();
    return GD_OK;
}

// The way of a frame over PCIe and its copy take 4.2 us each (four threads copying): one behind the other 48 frames are 0.4 ms, side by side little more than
// half of that.  The threads are begun when the first part has come, so that they wait for the others' way only, each for the part it is at.
int gd_expand_rgb24_pieces(const uint8_t *indexed, int32_t rows, const uint8_t *playpal, int32_t lane_count, int32_t part, uint8_t *staging, void *const *targets,
                           void *stream) {
    if (rows <= 0 || lane_count < 0 || part <= 0) return gd_fail(GD_E_ARG, "bad shape");
    if (lane_count == 0) return GD_OK;
    if (!indexed || !playpal || !staging || !targets) return gd_fail(GD_E_ARG, "null argument");
    for (int32_t k = 0; k < lane_count; ++k) if (!targets[k]) return gd_fail(GD_E_ARG, "null target");
    part = std::min(part, lane_count);    // any number above stands for all of them
    const size_t pixels = (size_t)rows * GD_SCREEN_WIDTH, bytes = pixels * 3;
    struct Events {                       // given back whatever happens
        std::vector<hipEvent_t> of;
        ~Events() { for (hipEvent_t event : of) (void)hipEventDestroy(event); }
    } events;
    int device = 0;
    GD_HIP_TRY(hipGetDevice(&device));
    int status = GD_OK;
    try {
        events.of.reserve((size_t)((lane_count - 1) / part + 1));
        for (int32_t first = 0; first < lane_count && status == GD_OK; first += part) {
            const int32_t count = std::min(part, lane_count - first);
            status = gd_expand_rgb24(indexed + (size_t)first * pixels, rows, playpal, count, staging + (size_t)first * bytes, stream);
            hipEvent_t event = nullptr;
            if (status == GD_OK && hipEventCreateWithFlags(&event, hipEventDisableTiming) != hipSuccess) status = gd_fail(GD_E_HIP, "hipEventCreateWithFlags");
            if (status == GD_OK) {
                events.of.push_back(event);
                if (hipEventRecord(event, static_cast<hipStream_t>(stream)) != hipSuccess) status = gd_fail(GD_E_HIP, "hipEventRecord");
            }
        }
    } catch (const std::exception &) { status = gd_fail(GD_E_ARG, "out of host memory"); }
    if (status != GD_OK) { (void)hipStreamSynchronize(static_cast<hipStream_t>(stream)); return status; }     // no frame is written into `staging` any more
    std::atomic<bool> failed{hipEventSynchronize(events.of[0]) != hipSuccess};
    constexpr int THREADS = 4;
    auto copy = [&](int first) {
        if (hipSetDevice(device) != hipSuccess) failed = true;
        int32_t come = 0;                 // parts that have
        for (int32_t k = first; k < lane_count; k += THREADS) {
            for (; come <= k / part; ++come) if (hipEventSynchronize(events.of[come]) != hipSuccess) failed = true;
            std::memcpy(targets[k], staging + (size_t)k * bytes, bytes);
        }
    };
    std::thread helpers[THREADS - 1];
    for (int t = 1; t < THREADS; ++t) {
        try { helpers[t - 1] = std::thread(copy, t); } catch (const std::exception &) { copy(t); }   // no thread to be had
    }
    copy(0);
    for (std::thread &helper : helpers) if (helper.joinable()) helper.join();
    return failed ? gd_fail(GD_E_HIP, "hipEventSynchronize") : GD_OK;
}

}  // extern "C"
