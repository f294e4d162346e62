// Batch closest-hit and visibility queries (the parity entry points).
#include "device.h"
#include "scene.h"
#include "traverse.h"

namespace cupbr {

__global__ __launch_bounds__(kTraceBlock) void k_trace_closest(DevScene S, const float* __restrict__ rays, size_t n,
                                                               int32_t* __restrict__ obj, int32_t* __restrict__ tri,
                                                               float* __restrict__ tout, uint32_t* spill) {
    __shared__ uint32_t lds[kTraceLds * kTraceBlock];
    const size_t gtid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    LaneStack<kTraceLds> st{lds + threadIdx.x, kTraceBlock, spill ? spill + gtid : nullptr, (uint32_t)stride};
    for (size_t i = gtid; i < n; i += stride) {
        const float* r = rays + 6 * i;
        v3 o = mk(r[0], r[1], r[2]), d = mk(r[3], r[4], r[5]);
        TraceResult res;
        traverse<false>(S, o, d, 0.0f, st, res);
        int32_t ob, tr;
        hit_ids(S, res, ob, tr);
        obj[i] = ob;
        tri[i] = tr;
        tout[i] = res.t;
    }
}

// Tracing::traceVisibility: visible iff no valid hit with t <= distance
__global__ __launch_bounds__(kTraceBlock) void k_trace_visibility(DevScene S, const float* __restrict__ rays,
                                                                  const float* __restrict__ dist, size_t n,
                                                                  uint8_t* __restrict__ vis, uint32_t* spill) {
    __shared__ uint32_t lds[kTraceLds * kTraceBlock];
    const size_t gtid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    LaneStack<kTraceLds> st{lds + threadIdx.x, kTraceBlock, spill ? spill + gtid : nullptr, (uint32_t)stride};
    for (size_t i = gtid; i < n; i += stride) {
        const float* r = rays + 6 * i;
        v3 o = mk(r[0], r[1], r[2]), d = mk(r[3], r[4], r[5]);
        TraceResult res;
        bool occluded = traverse<true>(S, o, d, dist[i], st, res);
        vis[i] = occluded ? 0 : 1;
    }
}

// Small batches: kGroup lanes per ray (traverse_group), one wave per block. LDS: 64 (depth + 1) words.
template <bool kAny, uint32_t kGroup>
__global__ __launch_bounds__(64) void k_trace_group(DevScene S, const float* __restrict__ rays,
                                                    const float* __restrict__ dist, size_t n,
                                                    int32_t* __restrict__ obj, int32_t* __restrict__ tri,
                                                    float* __restrict__ tout, uint8_t* __restrict__ vis,
                                                    uint32_t words) {
    extern __shared__ uint32_t group_lds[];
    const uint32_t g = threadIdx.x / kGroup;
    const size_t i = (size_t)blockIdx.x * (64 / kGroup) + g;
    const bool valid = i < n;
    const float* r = rays + 6 * (valid ? i : 0);
    const v3 o = mk(r[0], r[1], r[2]), d = mk(r[3], r[4], r[5]);
    TraceResult res;
    const bool any = traverse_group<kAny, kGroup>(S, o, d, kAny ? dist[valid ? i : 0] : 0.0f, valid, group_lds + g * words, res);
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
    if (64 * (s->stack_entries + 3) * sizeof(uint32_t) > (size_t)3 * 65536) return 0;  // the stacks fit 64 KiB of LDS
    return n <= 8192 ? 64 : n <= 32768 ? 32 : n <= 163840 ? 16 : 0;
}

template <bool kAny>
static int trace_group_launch(uint32_t lanes, const cupbr_scene* s, const float* rays, const float* dist, size_t n,
                              int32_t* obj, int32_t* tri, float* t, uint8_t* vis, hipStream_t stream) {
    const uint32_t entries = (s->stack_entries - 1u) / 3u + 1u;  // depth + 1
    const dim3 grid((unsigned)((n * lanes + 63) / 64));
    const auto launch = [&](auto kernel, uint32_t group) {
        hipLaunchKernelGGL(kernel, grid, dim3(64), 64 * entries * sizeof(uint32_t), stream, s->dev, rays, dist, n, obj, tri,
                           t, vis, group * entries);
    };
    switch (lanes) {
        case 64: launch(k_trace_group<kAny, 64>, 64); break;
        case 32: launch(k_trace_group<kAny, 32>, 32); break;
        default: launch(k_trace_group<kAny, 16>, 16); break;
    }
    CUPBR_HIP_CHECK(hipGetLastError());
    return CUPBR_OK;
}

int trace_closest_launch(const cupbr_scene* s, const float* rays, size_t n, int32_t* obj, int32_t* tri, float* t,
                         uint32_t* spill, int blocks, hipStream_t stream) {
    if (const uint32_t lanes = group_lanes(s, n))
        return trace_group_launch<false>(lanes, s, rays, nullptr, n, obj, tri, t, nullptr, stream);
    hipLaunchKernelGGL(k_trace_closest, dim3(blocks), dim3(kTraceBlock), 0, stream, s->dev, rays, n, obj, tri, t, spill);
    CUPBR_HIP_CHECK(hipGetLastError());
    return CUPBR_OK;
}

static int trace_grid(cupbr_scene* s, size_t n, uint32_t** spill) {
    int blocks = (int)std::min<size_t>((n + kTraceBlock - 1) / kTraceBlock, (size_t)device_cu_count() * 16);
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
    hipLaunchKernelGGL(k_trace_visibility, dim3(blocks), dim3(kTraceBlock), 0, stream, s->dev, rays, dist, n, vis, spill);
    CUPBR_HIP_CHECK(hipGetLastError());
    return scene_stream_release(s, stream);
}

}  // namespace cupbr
