// Batch closest-hit and visibility queries (the parity entry points).
#include "device.h"
#include "scene.h"
#include "traverse.h"

namespace cupbr {

// A wave's rays of a batch: pieces of `piece` consecutive ones, a grid's waves apart.
struct BatchShare {
    size_t base, n, stride;
    uint32_t piece, at, end;
    __device__ __forceinline__ void begin(size_t count, uint32_t size) {
        constexpr uint32_t kWaves = kTraceBlock / 64;
        n = count;
        piece = size;
        stride = (size_t)gridDim.x * kWaves * piece;
        base = ((size_t)blockIdx.x * kWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * piece;
        at = 0;
        end = base < n ? (uint32_t)min((size_t)piece, n - base) : 0u;
    }
    __device__ __forceinline__ bool refill() {
        base += stride;
        at = 0;
        end = base < n ? (uint32_t)min((size_t)piece, n - base) : 0u;
        return end != 0u;
    }
    __device__ __forceinline__ size_t index(uint32_t k) const { return base + k; }
};

__global__ __launch_bounds__(kTraceBlock) void k_trace_closest(DevScene S, const float* __restrict__ rays, size_t n,
                                                               int32_t* __restrict__ obj, int32_t* __restrict__ tri,
                                                               float* __restrict__ tout, uint32_t* spill, uint32_t piece) {
    __shared__ uint32_t lds[kTraceLds * kTraceBlock];
    const size_t gtid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    LaneStack<kTraceLds> st{lds + threadIdx.x, kTraceBlock, spill ? spill + gtid : nullptr, gridDim.x * blockDim.x};
    BatchShare share;
    share.begin(n, piece);
    trace_pool<false, false>(
        S, share, st,
        [&](size_t i, v3& o, v3& d, float& dist) {
            const float* r = rays + 6 * i;
            o = mk(r[0], r[1], r[2]);
            d = mk(r[3], r[4], r[5]);
            dist = 0.0f;
        },
        [&](size_t i, bool, const TraceResult& res) {
            int32_t ob, tr;
            hit_ids(S, res, ob, tr);
            obj[i] = ob;
            tri[i] = tr;
            tout[i] = res.t;
        });
}

// Tracing::traceVisibility: visible iff no valid hit with t <= distance
__global__ __launch_bounds__(kTraceBlock) void k_trace_visibility(DevScene S, const float* __restrict__ rays,
                                                                  const float* __restrict__ dist, size_t n,
                                                                  uint8_t* __restrict__ vis, uint32_t* spill,
                                                                  uint32_t piece) {
    __shared__ uint32_t lds[kTraceLds * kTraceBlock];
    const size_t gtid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    LaneStack<kTraceLds> st{lds + threadIdx.x, kTraceBlock, spill ? spill + gtid : nullptr, gridDim.x * blockDim.x};
    BatchShare share;
    share.begin(n, piece);
    trace_pool<true, false>(
        S, share, st,
        [&](size_t i, v3& o, v3& d, float& far) {
            const float* r = rays + 6 * i;
            o = mk(r[0], r[1], r[2]);
            d = mk(r[3], r[4], r[5]);
            far = dist[i];
        },
        [&](size_t i, bool occluded, const TraceResult&) { vis[i] = occluded ? 0 : 1; });
}

// Small batches: kGroup lanes per ray (trace_group), one wave per block.
constexpr uint32_t kGroupWords = 16;  // of the stacks, per lane
template <bool kAny, uint32_t kGroup>
__global__ __launch_bounds__(64) void k_trace_group(DevScene S, const float* __restrict__ rays,
                                                    const float* __restrict__ dist, size_t n,
                                                    int32_t* __restrict__ obj, int32_t* __restrict__ tri,
                                                    float* __restrict__ tout, uint8_t* __restrict__ vis) {
    __shared__ uint32_t lds[64 * kGroupWords];
    const uint32_t g = threadIdx.x / kGroup;
    const size_t i = (size_t)blockIdx.x * (64 / kGroup) + g;
    const bool valid = i < n;
    const float* r = rays + 6 * (valid ? i : 0);
    const v3 o = mk(r[0], r[1], r[2]), d = mk(r[3], r[4], r[5]);
    TraceResult res;
    uint32_t* stack = lds + g * kGroup * kGroupWords;
    const bool any = trace_group<kAny, kGroup, kGroup * kGroupWords>(
        S, o, d, kAny ? dist[valid ? i : 0] : 0.0f, valid, S.stack_reserve, [&](uint32_t k) -> uint32_t& { return stack[k]; }, res);
    if (!valid || threadIdx.x % kGroup) return;
    if (kAny) {
        vis[i] = any ? 0 : 1;
    } else {
        int32_t ob, tr;
        hit_ids(S, res, ob, tr);
        obj[i] = ob;
        tri[i] = tr;
        tout[i] = res.t;
    }
}

// Lanes per ray for a batch of n rays (0: one, with the kernels above): as many as the chip has idle. Closest
// hit, us, in a scene of overlapping meshes / one of spheres and boxes, with 64, 32, 16 lanes a ray and one:
//   2048 rays     23 / 15     32 / 17     50 / 18    324 / 64
//   8192 rays     34 / 22     42 / 19     55 / 20    340 / 68
//   32768 rays    72 / 42     69 / 33     77 / 26    318 / 70
//   131072 rays  231 / 129   188 / 82    186 / 58    307 / 70
//   262144 rays  447 / 244   361 / 152   337 / 102   379 / 95
// Visibility lies alike (2048 rays 19 / 17 with 64 lanes, 165 / 41 with one; 163840 rays 121 / 57 with 16,
// 184 / 61 with one).
static uint32_t group_lanes(const cupbr_scene* s, size_t n) {
    if (s->stack_entries > 16 * kGroupWords) return 0;  // the smallest group's stack
    return n <= 8192 ? 64 : n <= 32768 ? 32 : n <= 163840 ? 16 : 0;
}

template <bool kAny>
static int trace_group_launch(uint32_t lanes, const cupbr_scene* s, const float* rays, const float* dist, size_t n,
                              int32_t* obj, int32_t* tri, float* t, uint8_t* vis, hipStream_t stream) {
    const dim3 grid((unsigned)((n * lanes + 63) / 64));
    const auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(64), 0, stream, s->dev, rays, dist, n, obj, tri, t, vis);
    };
    if (lanes == 64)
        launch(k_trace_group<kAny, 64>);
    else if (lanes == 32)
        launch(k_trace_group<kAny, 32>);
    else
        launch(k_trace_group<kAny, 16>);
    CUPBR_HIP_CHECK(hipGetLastError());
    return CUPBR_OK;
}

// Rays of a wave's piece: the batch over 4096 waves (4 per SIMD), so that the waves run side by side and refill
// their lanes as often as that leaves them rays; the longest ray of a batch that fits the chip bounds it. With
// 8192 and 2560 waves 1 M rays (overlapping meshes) took 940 and 1198 us, with 4096 848 (and 778 with a
// refill at 16 idle lanes instead of 32); 64 rays per wave and no refill 1184. Spheres and boxes: 2 M rays
// 477 -> 341 us, 1 M 447 -> 253, 262144 91 -> 77. Lanes per vector instruction 11 -> 24.
static uint32_t batch_piece(size_t n) {
    return (uint32_t)std::min<size_t>(std::max<size_t>((n / 4096 + 63) & ~(size_t)63, 64), 512);
}
static size_t batch_blocks(size_t n) {
    const size_t rays = (size_t)batch_piece(n) * (kTraceBlock / 64);
    return (n + rays - 1) / rays;
}

int trace_closest_launch(const cupbr_scene* s, const float* rays, size_t n, int32_t* obj, int32_t* tri, float* t,
                         uint32_t* spill, int blocks, hipStream_t stream) {
    if (const uint32_t lanes = group_lanes(s, n))
        return trace_group_launch<false>(lanes, s, rays, nullptr, n, obj, tri, t, nullptr, stream);
    blocks = (int)std::min<size_t>(blocks, batch_blocks(n));
    hipLaunchKernelGGL(k_trace_closest, dim3(blocks), dim3(kTraceBlock), 0, stream, s->dev, rays, n, obj, tri, t, spill,
                       batch_piece(n));
    CUPBR_HIP_CHECK(hipGetLastError());
    return CUPBR_OK;
}

static int trace_grid(cupbr_scene* s, size_t n, uint32_t** spill) {
    int blocks = (int)std::min<size_t>(batch_blocks(n), (size_t)device_cu_count() * 16);
    blocks = std::max(blocks, 1);
    *spill = nullptr;
    if (!group_lanes(s, n) && s->stack_entries > (uint32_t)kTraceLds) {
        size_t need = (size_t)(s->stack_entries - kTraceLds) * blocks * kTraceBlock * sizeof(uint32_t);
        int rc = s->spill.ensure(need);
        if (rc) return -1;
        *spill = s->spill.as<uint32_t>();
    }
    return blocks;
}

int trace_closest_device(const cupbr_scene* cs, const float* rays, size_t n, int32_t* obj, int32_t* tri, float* t,
                         hipStream_t stream) {
    if (n == 0) return CUPBR_OK;
    cupbr_scene* s = const_cast<cupbr_scene*>(cs);
    if (int rc = scene_upload(s)) return rc;
    uint32_t* spill;
    if (int rc = scene_stream_acquire(s, stream)) return rc;
    int blocks = trace_grid(s, n, &spill);
    if (blocks < 0) return CUPBR_ERR_OUT_OF_MEMORY;
    if (int rc = trace_closest_launch(s, rays, n, obj, tri, t, spill, blocks, stream)) return rc;
    return scene_stream_release(s, stream);
}

int trace_visibility_device(const cupbr_scene* cs, const float* rays, const float* dist, size_t n, uint8_t* vis,
                            hipStream_t stream) {
    if (n == 0) return CUPBR_OK;
    cupbr_scene* s = const_cast<cupbr_scene*>(cs);
    if (int rc = scene_upload(s)) return rc;
    uint32_t* spill;
    if (int rc = scene_stream_acquire(s, stream)) return rc;
    int blocks = trace_grid(s, n, &spill);
    if (blocks < 0) return CUPBR_ERR_OUT_OF_MEMORY;
    if (const uint32_t lanes = group_lanes(s, n)) {
        if (int rc = trace_group_launch<true>(lanes, s, rays, dist, n, nullptr, nullptr, nullptr, vis, stream)) return rc;
        return scene_stream_release(s, stream);
    }
    hipLaunchKernelGGL(k_trace_visibility, dim3(blocks), dim3(kTraceBlock), 0, stream, s->dev, rays, dist, n, vis, spill,
                       batch_piece(n));
    CUPBR_HIP_CHECK(hipGetLastError());
    return scene_stream_release(s, stream);
}

}  // namespace cupbr
