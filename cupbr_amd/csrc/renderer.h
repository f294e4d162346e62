// Host-side renderer handle (cupbr_renderer): PBRenderer's state
// (lib/src/Renderer/PBRenderer.cu:26-52) plus the wavefront buffers.
#pragma once

#include <vector>

#include "device.h"
#include "nrc.h"
#include "scene.h"

namespace cupbr {

constexpr int kNumImages = 8;  // cupbr_image

// Device counters of one render call, one 128-byte line each so that atomics on
// different counters never serialise on the same L2 line. The trace kernel's work
// counters hand out pieces of an XCD's rays to its persistent waves; each counter is reset by
// the kernel that runs after its last user.
struct alignas(128) CounterLine {
    uint32_t v;
    uint32_t pad[31];
};
// the extension and shadow rays that one XCD's blocks made at a bounce
struct alignas(128) RayCount {
    union {
        struct {
            uint32_t ext, shadow;
        };
        unsigned long long both;
    };
    uint32_t pad[30];
};
// The ray queues of a batch, cut into granules of 2^lg slots: granule k belongs to XCD k % 8 (the blocks b
// with b % 8 = k % 8). An XCD appends to its own granules, in order, the rays that its blocks shade, and
// traces and shades those: every counter and most queue lines stay in one L2, and the XCDs keep equal
// shares of the image without taking rays from each other. (One counter for all, an add of 13 ns per 256
// rays and queue, was a part of every shade: 5.26 -> 4.74 ms for the first one of 133 M paths; gradient domain
// 7.40 -> 6.83 ms, mixed primitives, 331x217, 6 spp, 407 -> 385 us.) A path stays on its
// XCD, so an XCD's queue never outgrows the paths it began with.
struct XcdQueue {
    uint32_t lg;
    // slot of XCD x's ray r
    __host__ __device__ uint32_t slot(uint32_t x, uint32_t r) const {
        return ((r >> lg) * 8u + x) << lg | (r & ((1u << lg) - 1u));
    }
    // XCD x's rays of a queue whose first n slots are filled
    __host__ __device__ uint32_t length(uint32_t n, uint32_t x) const {
        const uint32_t whole = n >> (lg + 3u), rest = n - (whole << (lg + 3u)), skip = x << lg, g = 1u << lg;
        return (whole << lg) + (rest > skip ? (rest - skip < g ? rest - skip : g) : 0u);
    }
    // slots that hold n rays
    __host__ __device__ uint32_t capacity(uint32_t n) const { return (n + (8u << lg) - 1u) >> (lg + 3u) << (lg + 3u); }
};
struct Counters {
    RayCount rays[2][8];         // by the parity of the bounce that made them, per XCD
    CounterLine inside[2][8];    // volume renderer: rays inside an object, likewise
    CounterLine work[8];         // trace kernel: extension rays handed out beyond the dealt pieces, per XCD
    CounterLine swork[8];        // trace kernel: shadow rays handed out beyond the dealt pieces, per XCD
    union alignas(128) CacheCount {
        struct {
            uint32_t queries, rows;  // radiance-cache queries and training rows of the batch
        };
        unsigned long long both;
    } cache;
    CacheCount cache_part[8];    // whole paths: those of each XCD's blocks
    CounterLine query_early;  // queries that existed after the second bounce's shade
    unsigned long long extension_rays;
    unsigned long long shadow_rays;
    unsigned long long ext_nodes, ext_prims, shadow_nodes, shadow_prims;  // traversal counting
    unsigned long long refill_launches;  // trace launches that handed rays to idle lanes
    unsigned long long cache_queries, cache_rows;  // radiance-cache queries and training rows of the call
};

// HIP events recorded between consecutive launches on the renderer's stream;
// stage time = time between the event before a launch and the event after it
struct StageTimer {
    std::vector<hipEvent_t> pool;
    std::vector<int> stage;  // stage[i]: stage of the launch that ends at event i (-1: first event)
    size_t used = 0;
    int mark(hipStream_t st, int s) {
        if (used == pool.size()) {
            hipEvent_t e;
            if (hipEventCreate(&e) != hipSuccess) return CUPBR_ERR_HIP;
            pool.push_back(e);
            stage.push_back(-1);
        }
        stage[used] = s;
        if (hipEventRecord(pool[used], st) != hipSuccess) return CUPBR_ERR_HIP;
        ++used;
        return CUPBR_OK;
    }
    ~StageTimer() {
        for (hipEvent_t e : pool) (void)hipEventDestroy(e);
    }
};

struct Wavefront {
    uint32_t capacity = 0;  // paths
    DevBuf weight;          // float4 per path: throughput.xyz, rng state (bits)
    DevBuf radiance;        // float4 per path
    DevBuf q_o[2], q_d[2];  // float4 per entry: origin | direction.xyz, path (bits)
    DevBuf q_hit;           // float2 per entry: t, prim (bits)
    DevBuf s_o[2], s_d[2], s_c[2];  // shadow queues by bounce parity: origin.xyz+distance |
                                    // direction.xyz+path | contribution
    DevBuf counters;
    DevBuf spill;
    DevBuf gdpt_slot;  // gradient-domain groups: queue slot of the base path's ray, by bounce parity
    DevBuf iq_o[2], iq_d[2];  // volume renderer: rays inside an object (traced against that object)
    uint32_t iq_capacity = 0;
    uint32_t spill_entries = 0;
};

}  // namespace cupbr

struct cupbr_renderer {
    int32_t method = CUPBR_RAYTRACER;
    uint32_t width = 0, height = 0;
    bool output_size_set = false;
    const cupbr_scene* scene = nullptr;
    uint32_t frame_index = 0;
    uint32_t max_trace_depth = 5;   // PBRenderer.cu:59
    bool russian_roulette = false;  // uninitialised in the reference (PBRenderer.cu:51); off here
    int32_t gdpt_mode = CUPBR_GDPT_TRIMMED_MEAN;  // reconstruction of GRADIENTDOMAIN frames
    int32_t rng = CUPBR_RNG_TEA_LCG;              // random numbers of PATHTRACER frames
    float gdpt_alpha = 0.2f;                      // screened-Poisson weight of the primal image
    uint32_t gdpt_iterations = 50;                // screened-Poisson Jacobi iterations
    cupbr::DevBuf images[cupbr::kNumImages];
    cupbr::DevBuf temp;
    cupbr::Wavefront wf;
    hipStream_t stream = nullptr;
    hipEvent_t ev_start = nullptr, ev_stop = nullptr;
    cupbr_render_stats stats{};
    bool profiling = false;
    bool counting = false;
    cupbr::StageTimer timer;
    // radiance cache (PATHTRACER only; nullptr = plain PT)
    cupbr_nrc* nrc = nullptr;
    uint32_t nrc_train_paths = 1u << 16;  // training paths per frame (full-length PT paths)
    uint32_t nrc_steps = 16;              // Adam steps per frame
    uint32_t nrc_batch = 1u << 14;        // rows per step
    float nrc_lr = 1e-3f;
    float nrc_camera_min_roughness = __builtin_inff();  // camera-hit cache vertices (+inf: none)
    uint32_t nrc_max_rows = 1u << 18;     // training rows kept per frame
    cupbr::DevBuf nrc_queries, nrc_pending, nrc_rows;
    bool counted = false;  // the last cupbr_render call launched paths, and wf.counters holds its counts
    // second stream for cache inference that overlaps the training paths' later bounces
    hipStream_t side_stream = nullptr;
    hipEvent_t ev_queries = nullptr, ev_side_done = nullptr;
};

namespace cupbr {

int renderer_clear_images(cupbr_renderer* r);
// records a stage boundary when profiling is on (stage: 0 extend, 1 shade, 2 shadow, 3 other)
inline int stage_mark(cupbr_renderer* r, int stage) { return r->profiling ? r->timer.mark(r->stream, stage) : CUPBR_OK; }
// one reference frame per sample: frames [frame0, frame0+spp) of method PATHTRACER
int render_pathtracer(cupbr_renderer* r, const cupbr_camera& cam, uint32_t frame0, uint32_t spp);
int render_volume(cupbr_renderer* r, const cupbr_camera& cam, uint32_t frame0, uint32_t spp);
int render_gdpt(cupbr_renderer* r, const cupbr_camera& cam, uint32_t frame0, uint32_t spp);
// the gradient-domain paths of frames [frame0, frame0+spp) in wavefront form: running means of the
// base and the four gradient buffers (pathtracer.hip)
int gdpt_paths_wavefront(cupbr_renderer* r, const cupbr_camera& cam, uint32_t frame0, uint32_t spp);
// the volume renderer's frames [frame0, frame0+spp) in wavefront form (pathtracer.hip)
int volume_paths_wavefront(cupbr_renderer* r, const cupbr_camera& cam, uint32_t frame0, uint32_t spp);
int render_raytracer(cupbr_renderer* r, const cupbr_camera& cam);

}  // namespace cupbr
