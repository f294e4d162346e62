// PT+NEE in wavefront form (pathtracer_kernel_nee, lib/src/Renderer/PathTracer.cu:97-169).
//
// Per batch of paths (one path = one pixel of one reference frame):
//   camera      the camera rays, made and traced as wave packets       (PathTracer.cu:112-126)
//   per bounce: trace    (from bounce 1 on) closest hit for the bounce's extension rays (:126), and any-hit
//                        visibility for the previous bounce's shadow rays, adding their
//                        NEE terms (:64-73), in one launch
//               shade    emission, NEE sample -> shadow queue,         (:127-158)
//                        Russian roulette, BSDF sample -> next extension queue
//   final trace the last bounce's shadow rays
//   accumulate  the reference running mean, frame by frame             (:162-168)
// A small batch runs its paths whole in one launch instead (k_pt_paths), then accumulate. Where the camera rays
// cannot be packets (the visit-counting pass, no tree, a tree deeper than the packets' stack), raygen writes them
// into extension queue 0 and bounce 0 is a trace like the others.
// Queue lengths live on the device, so no host round trip happens between bounces.
// trace is a persistent grid whose waves take pieces of their XCD's rays from its work counter
// (traversal cost varies per ray; one launch per bounce keeps the GPU full
// where the shadow queue alone is short); shade walks its queue with a static grid stride and
// appends to the next queues with one atomic per 256-entry block (ballot + LDS prefix).
// Extension and shadow queues alternate by bounce parity.
//
// Differences from the reference that cannot change the image: a path whose
// throughput became exactly zero (back-facing hit, :36-41) stops instead of
// bouncing on with zero weight, and a shadow ray whose contribution is exactly
// zero is not traced.
#include "renderer.h"
#include "shading.h"
#include "traverse.h"

// Rays per lane of the persistent grid from which a trace launch refills its lanes; below, every wave
// traces one 64-ray chunk, whose end waits for one tail, not for two (extension rays, then shadow
// rays). 1080p / 1M triangles at 1 spp with 1, 2 and 4 rays: 4.00, 4.09 and 4.27 ms (the volume renderer,
// 512x512, 16 spp: 2.63, 2.62, 2.58).
#ifndef CUPBR_REFILL_MIN
#define CUPBR_REFILL_MIN 1u
#endif

namespace cupbr {

constexpr int kPtBlock = 256;
constexpr int kPtWaves = kPtBlock / 64;
// traversal stack entries per lane kept in LDS (16 KB per 256-thread block: the trace kernel's 63
// VGPRs, not LDS, then bound its occupancy at 8 waves per SIMD; deeper entries spill to memory)
constexpr int kPtLds = 16;
// Batches of up to this many paths per CU run whole paths in one launch (k_pt_paths): as many as plain frames have
// resident at once with 64 paths a wave (113 VGPRs, 4 waves per SIMD; the 8-lane walk takes 144, 3 waves, and with
// the cache 192, 2 waves). What bounds a small batch is the longest path's chain of rays and, with a launch and a
// queue per bounce, the launches; a resident batch needs neither queues nor the path state in memory. Frames of
// 256x256, 1 spp, depth 5, queues / whole paths (us): spheres and boxes 819 / 277, 1M triangles 1503 / 761; 512x512:
// 994 / 590, 1623 / 1541. At 331x217, 6 spp (1.6 times the limit) 1003 / 738, but 1786 / 2371.
constexpr uint32_t kWholePaths = 1024;
// Traversal stack entries (three per BVH4 level) above which a wave of such a batch holds only as many paths (8 to 32)
// as 16 waves per CU need, so that 8 lanes walk the tree for each: 1M triangles, 64x64, 1 spp, 1310 -> 312 us, 256x256
// 1318 -> 761. In a shallow tree that pays up to 64 paths per CU only (Cornell box, depth 5: 64x64 158 -> 100 us, but
// 256x256 156 -> 225); beyond it a wave takes 64 paths.
constexpr uint32_t kDeepStack = 24;
// The limits of plain frames in a shallow tree, of more bounces than one and of one. There the queues' launches end
// sooner, so that they catch up where the waves of whole paths no longer all start at once (us, queues / whole paths;
// Cornell box, mixed primitives, spheres and boxes):
//   depth 2:  160x160 84 / 71, 88 / 67, 71 / 55;  256x255 85 / 78, 88 / 68, 71 / 63;  362x362 89 / 94, 93 / 91, 71 / 83
//   depth 5:  160x160 158 / 150, 184 / 146, 116 / 97;  256x255 160 / 147, 175 / 146, 118 / 102;
//             362x362 170 / 163, 181 / 156, 122 / 113;  512x256 165 / 159, 182 / 153, 119 / 124
//   depth 1:  200x200 52 / 50, 52 / 47, 44 / 44;  256x255 52 / 59, 53 / 54, 44 / 52
constexpr uint32_t kWholeShallow = 256, kWholeShallowDirect = 192;

// Block-wide append: every thread of the block calls it; lanes with `want` get consecutive
// slots of the queue whose length is *count (one atomic per block).
__device__ __forceinline__ uint32_t block_append(bool want, uint32_t* count, uint32_t* s) {
    const unsigned long long m = __ballot(want);
    const uint32_t wave = threadIdx.x >> 6, lane = __lane_id();
    if (lane == 0) s[wave] = (uint32_t)__popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t tot = 0;
        for (int w = 0; w < kPtWaves; ++w) {
            const uint32_t c = s[w];
            s[w] = tot;
            tot += c;
        }
        s[kPtWaves] = tot ? atomicAdd(count, tot) : 0u;
    }
    __syncthreads();
    const uint32_t slot = s[kPtWaves] + s[wave] + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
    __syncthreads();
    return slot;
}

// block_append to two queues together: one 64-bit add for both counts (the low and the high word of
// *count). s: 2 (kPtWaves + 1) words.
__device__ __forceinline__ void block_append2(bool want_lo, bool want_hi, unsigned long long* count, uint32_t* s,
                                              uint32_t& lo, uint32_t& hi) {
    const unsigned long long me = __ballot(want_lo), ms = __ballot(want_hi);
    const uint32_t wave = threadIdx.x >> 6, lane = __lane_id();
    if (lane == 0) {
        s[2 * wave] = (uint32_t)__popcll(me);
        s[2 * wave + 1] = (uint32_t)__popcll(ms);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long tot = 0;
        for (int w = 0; w < kPtWaves; ++w) {
            const uint32_t e = s[2 * w], h = s[2 * w + 1];
            s[2 * w] = (uint32_t)tot;
            s[2 * w + 1] = (uint32_t)(tot >> 32);
            tot += (unsigned long long)h << 32 | e;
        }
        const unsigned long long base = tot ? atomicAdd(count, tot) : 0ull;
        s[2 * kPtWaves] = (uint32_t)base;
        s[2 * kPtWaves + 1] = (uint32_t)(base >> 32);
    }
    __syncthreads();
    const unsigned long long below = (1ull << lane) - 1ull;
    lo = s[2 * kPtWaves] + s[2 * wave] + (uint32_t)__popcll(me & below);
    hi = s[2 * kPtWaves + 1] + s[2 * wave + 1] + (uint32_t)__popcll(ms & below);
    __syncthreads();
}

// adds a wave's traversal counts to two device counters
__device__ __forceinline__ void wave_add_counts(const TravCount& tc, unsigned long long* nodes,
                                                unsigned long long* prims) {
    unsigned long long a = tc.nodes, b = tc.prims;
    for (int off = 32; off > 0; off >>= 1) {
        a += __shfl_xor(a, off);
        b += __shfl_xor(b, off);
    }
    if (__lane_id() == 0) {
        atomicAdd(nodes, a);
        atomicAdd(prims, b);
    }
}

__device__ __forceinline__ uint32_t hash32(uint32_t x) {
    x ^= x >> 16;
    x *= 0x7feb352du;
    x ^= x >> 15;
    x *= 0x846ca68bu;
    x ^= x >> 16;
    return x;
}

// radiance-cache training paths: pixel/frame pairs whose hash falls below the threshold
__device__ __forceinline__ bool is_training_path(uint32_t pix, uint32_t frame, uint32_t thresh) {
    return thresh != 0u && hash32(pix * 0x9E3779B1u ^ hash32(frame + 0x632BE5ABu)) < thresh;
}

// rad[p].w carries the path's flags: bit 0 = radiance-cache training path
// a path's first generator state: the reference's tea<4>(pixel, frame) (PathTracer.cu:112), or for
// the PCG mode the PCG hash of the pixel keyed by the hash of the frame
template <class Seed> __device__ __forceinline__ Seed path_seed(uint32_t pix, uint32_t frame);
template <> __device__ __forceinline__ uint32_t path_seed<uint32_t>(uint32_t pix, uint32_t frame) {
    return tea4(pix, frame);
}
template <> __device__ __forceinline__ Pcg32 path_seed<Pcg32>(uint32_t pix, uint32_t frame) {
    return Pcg32{pcg_hash(pcg_hash(frame) ^ pix)};
}

// The camera ray of queue slot p of a batch in SampleOrder (PathTracer.cu:112-126): the pixel it
// samples, frame frame0 + its sample index, and the generator state after launchRay's two draws.
template <class Seed>
__device__ __forceinline__ void camera_path(const cupbr_camera& cam, uint32_t w, uint32_t h, uint32_t frame0,
                                            const SampleOrder& order, uint32_t p, Seed& seed, uint32_t& pix,
                                            uint32_t& frame, v3& o, v3& d) {
    uint32_t s, j, px, py;
    order.sample(p, s, j);
    tile_pixel(j, w, h, px, py);
    pix = py * w + px;
    frame = frame0 + s;
    seed = path_seed<Seed>(pix, frame);
    launch_ray(px, py, w, h, cam, seed, o, d);
}

// the per-batch counter reset that precedes bounce 0 (whose rays are those of parity 1), by threads 0..7
// of the calling kernel's first block: thread x for XCD x
__device__ __forceinline__ void reset_batch_counters(Counters* c, XcdQueue order, uint32_t npath, uint32_t x) {
    c->rays[1][x].ext = order.length(npath, x);
    c->rays[1][x].shadow = 0;
    c->rays[0][x].both = 0;
    c->work[x].v = c->swork[x].v = 0;
    c->inside[0][x].v = c->inside[1][x].v = 0;
    if (x == 0) c->cache.both = 0;
}

// A camera path's state as bounce 0 leaves it: direction and path id (queue 0), throughput 1 and
// generator state, radiance 0 and flags (bit 0: radiance-cache training path).
template <class Seed>
__device__ __forceinline__ void store_camera_path(uint32_t p, v3 d, Seed seed, uint32_t pix, uint32_t frame,
                                                  uint32_t train_thresh, float4* __restrict__ q_d,
                                                  float4* __restrict__ weight, float4* __restrict__ rad) {
    q_d[p] = make_float4(d.x, d.y, d.z, __uint_as_float(p));
    weight[p] = make_float4(1.0f, 1.0f, 1.0f, __uint_as_float(state_bits(seed)));
    const uint32_t flags = is_training_path(pix, frame, train_thresh) ? 1u : 0u;
    rad[p] = make_float4(0.0f, 0.0f, 0.0f, __uint_as_float(flags));
}

// Camera rays of a batch in SampleOrder: the path id of a path is its queue slot here.
template <class Seed>
__global__ __launch_bounds__(kPtBlock) void k_pt_raygen(cupbr_camera cam, uint32_t w, uint32_t h, uint32_t frame0,
                                                        uint32_t npath, SampleOrder order, float4* __restrict__ q_o,
                                                        float4* __restrict__ q_d, float4* __restrict__ weight,
                                                        float4* __restrict__ rad, Counters* c, XcdQueue queue,
                                                        uint32_t train_thresh) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < 8) reset_batch_counters(c, queue, npath, p);
    if (p >= npath) return;  // p: queue slot and path id
    Seed seed;
    uint32_t pix, frame;
    v3 o, d;
    camera_path(cam, w, h, frame0, order, p, seed, pix, frame, o, d);
    q_o[p] = make_float4(o.x, o.y, o.z, 0.0f);
    store_camera_path(p, d, seed, pix, frame, train_thresh, q_d, weight, rad);
}

// paths of a batch from which the cache is asked on a second stream while the later bounces are traced
// (for a 256x256 frame the extra launches and stream waits cost more than the 7 us that they hide)
constexpr uint32_t kSidePaths = 1u << 20;

// radiance-cache records written by shade: a query (inputs 16, throughput 3, path) ends a rendering
// path at its first diffuse/glossy vertex after the camera hit; a training path leaves a pending
// row (inputs 16, radiance so far 3, throughput 3, path, pad) at each such vertex
struct NrcShade {
    float4* queries;  // 5 float4 per query
    float4* pending;  // 6 float4 per row
    uint32_t max_rows;
    // the camera hit is also a cache vertex when its material is Lambertian or GGX with roughness
    // >= camera_min_roughness (+inf: never)
    float camera_min_roughness;
};

// What a path's vertex adds and asks for.
struct Vertex {
    bool emits, next, shadow, query, row;
    v3 emission;  // to the path's radiance (emits), before the light's contribution
    v3 next_o, next_d;
    v3 shadow_o, shadow_d, light;  // shadow ray, and what the light adds if it is visible
    float dist;
    float4 rec[6];  // cache query or pending row
};

// One vertex of path p, where its ray (o, d) hit prim at t, or left the scene: PathTracer.cu:20-160 in the
// reference's order. w3: throughput. L: the path's radiance so far, for the cache's records only.
template <bool kNrc, class Seed>
__device__ __forceinline__ void path_vertex(const DevScene& S, uint32_t bounce, uint32_t max_depth, int rr,
                                            const NrcShade& nrc, v3 o, v3 d, float t, uint32_t prim, uint32_t p,
                                            bool training, v3 L, v3& w3, Seed& seed, Vertex& v) {
    v.emits = v.next = v.shadow = v.query = v.row = false;
    if (prim == kNoHit) {  // :127-135
        if (S.use_env) {
            v.emission = w3 * env_lookup(S, d);
            v.emits = true;
        }
        return;
    }
    const float nl = (float)(S.n_lights + (S.use_env ? 1u : 0u));
    const v3 P = o + t * d;  // geom.P = origin + t * direction
    v3 N;
    uint32_t obj;
    hit_geometry(S, prim, P, N, obj);
    const Mat m = load_mat(S.mats + obj);
    const v3 inc = -1.0f * d;
    // emissiveIllumintation :20-26; nothing for a black surface, unless the throughput is infinite or NaN
    v.emission = w3 * m.albedo_e;
    v.emits = !(v.emission.x == 0.0f && v.emission.y == 0.0f && v.emission.z == 0.0f);
    const bool cache_vertex = bounce >= 1 ? (m.type == CUPBR_LAMBERT || m.type == CUPBR_PHONG || m.type == CUPBR_GGX)
                                          : ((m.type == CUPBR_LAMBERT && nrc.camera_min_roughness <= 1.0f) ||
                                             (m.type == CUPBR_GGX && m.roughness >= nrc.camera_min_roughness));
    if (kNrc && cache_vertex && !(dot(N, inc) <= 0.0f)) {
        v.rec[0] = make_float4(P.x, P.y, P.z, inc.x);
        v.rec[1] = make_float4(inc.y, inc.z, N.x, N.y);
        v.rec[2] = make_float4(N.z, m.roughness, m.albedo_d.x, m.albedo_d.y);
        v.rec[3] = make_float4(m.albedo_d.z, m.albedo_s.x, m.albedo_s.y, m.albedo_s.z);
        if (!training) {  // rendering path: ends here with throughput * cache
            v.query = true;
            v.rec[4] = make_float4(w3.x, w3.y, w3.z, __uint_as_float(p));
            return;
        }
        v.row = true;  // training path: pending row, the path goes on
        L += v.emission;
        v.rec[4] = make_float4(L.x, L.y, L.z, w3.x);
        v.rec[5] = make_float4(w3.y, w3.z, __uint_as_float(p), 0.0f);
    }
    if (m.type != CUPBR_GLASS && dot(N, inc) <= 0.0f) return;  // :36-41
    // directIllumination :43-73
    v3 ldir, le;
    float dist = 0.0f;
    if (nee_sample(S, m, seed, P, inc, N, ldir, le, dist)) {
        v.light = (nl * fmaxf(0.0f, dot(N, ldir))) * brdf(m, inc, ldir, N) * le * w3;
        if (!(v.light.x == 0.0f && v.light.y == 0.0f && v.light.z == 0.0f)) {
            v.shadow = true;
            v.shadow_o = P + 0.001f * ldir;
            v.shadow_d = normalize(ldir);
            v.dist = dist;
        }
    }
    if (rr) {  // :141-152
        const float alpha = clampf(fmaxf(w3.x, fmaxf(w3.y, w3.z)), 0.0f, 1.0f);
        if (rnd(seed) > alpha || safe_float_equal(alpha, 0.0f)) return;
        w3 = w3 / alpha;
    }
    // indirectIllumination :76-95
    const DirPdf sp = sample_direction(m, seed, inc, N);
    if (norm(sp.d) < kEpsilon) return;
    w3 = w3 * fabsf(dot(sp.d, N)) * brdf(m, inc, sp.d, N) / sp.pdf;
    if (bounce + 1 < max_depth) {  // :156-160
        v.next = true;
        v.next_o = P + 0.01f * sp.d;
        v.next_d = normalize(sp.d);
    }
}

template <bool kNrc, class Seed>
__device__ __forceinline__ void pt_shade(const DevScene& S, int cur, uint32_t bounce, uint32_t max_depth, int rr,
                                         const float4* __restrict__ q_o, const float4* __restrict__ q_d,
                                         const float2* __restrict__ q_hit, float4* __restrict__ nq_o,
                                         float4* __restrict__ nq_d, float4* __restrict__ s_o, float4* __restrict__ s_d,
                                         float4* __restrict__ s_c, float4* __restrict__ weight,
                                         float4* __restrict__ rad, Counters* c, XcdQueue queue, const NrcShade& nrc,
                                         uint32_t omask) {
    __shared__ uint32_t s_append[2 * (kPtWaves + 1)];
    const uint32_t xcd = blockIdx.x & 7u, n = c->rays[cur ^ 1][xcd].ext;
    if (blockIdx.x == 0 && threadIdx.x < 8)  // the next trace starts at 0
        c->work[threadIdx.x].v = c->swork[threadIdx.x].v = 0;
    for (uint32_t base = (blockIdx.x >> 3) * kPtBlock; base < n; base += (gridDim.x >> 3) * kPtBlock) {
        const uint32_t i = queue.slot(xcd, base + threadIdx.x);
        Vertex v;
        v.next = v.shadow = v.query = v.row = false;
        uint32_t p = 0;
        if (base + threadIdx.x < n) {
            const float4 o4 = q_o[i & omask], d4 = q_d[i];
            const float2 hh = q_hit[i];
            const bool first = omask == 0u;
            p = first ? i : __float_as_uint(d4.w);
            const float4 W = first ? make_float4(1.0f, 1.0f, 1.0f, d4.w) : weight[p];
            float4 R = {};
            if (kNrc) R = rad[p];
            v3 w3 = mk(W.x, W.y, W.z);
            Seed seed = seed_from_bits<Seed>(__float_as_uint(W.w));
            path_vertex<kNrc, Seed>(S, bounce, max_depth, rr, nrc, mk(o4.x, o4.y, o4.z), mk(d4.x, d4.y, d4.z), hh.x,
                                    __float_as_uint(hh.y), p, __float_as_uint(R.w) & 1u, mk(R.x, R.y, R.z), w3, seed, v);
            if (v.emits) {
                if (!kNrc) R = rad[p];
                rad[p] = make_float4(R.x + v.emission.x, R.y + v.emission.y, R.z + v.emission.z, R.w);
            }
            if (v.next) weight[p] = make_float4(w3.x, w3.y, w3.z, __uint_as_float(state_bits(seed)));
        }
        uint32_t ns, ss;
        block_append2(v.next, v.shadow, &c->rays[cur][xcd].both, s_append, ns, ss);
        if (v.next) {
            ns = queue.slot(xcd, ns);
            nq_o[ns] = make_float4(v.next_o.x, v.next_o.y, v.next_o.z, 0.0f);
            nq_d[ns] = make_float4(v.next_d.x, v.next_d.y, v.next_d.z, __uint_as_float(p));
        }
        if (v.shadow) {
            ss = queue.slot(xcd, ss);
            s_o[ss] = make_float4(v.shadow_o.x, v.shadow_o.y, v.shadow_o.z, v.dist);
            s_d[ss] = make_float4(v.shadow_d.x, v.shadow_d.y, v.shadow_d.z, __uint_as_float(p));
            s_c[ss] = make_float4(v.light.x, v.light.y, v.light.z, 0.0f);
        }
        if (kNrc) {
            uint32_t qs, rs;
            block_append2(v.query, v.row, &c->cache.both, s_append, qs, rs);
            if (v.query)
                for (int k = 0; k < 5; ++k) nrc.queries[(size_t)qs * 5 + k] = v.rec[k];
            if (v.row && rs < nrc.max_rows)
                for (int k = 0; k < 6; ++k) nrc.pending[(size_t)rs * 6 + k] = v.rec[k];
        }
    }
}

// Shade without the radiance cache. amdgpu_waves_per_eu(5, 8): 96 VGPRs instead of 102 and 5
// waves per SIMD instead of 4, without spills (23.7 -> 23.1 ms of shading per 1080p 64-spp step;
// 6 and 8 waves spill and are slower). The cache variant keeps its 145 VGPRs, 3 waves (it would spill).
template <class Seed>
__global__ __launch_bounds__(kPtBlock) __attribute__((amdgpu_waves_per_eu(5, 8)))
void k_pt_shade(DevScene S, int cur, uint32_t bounce, uint32_t max_depth, int rr, const float4* __restrict__ q_o,
                const float4* __restrict__ q_d, const float2* __restrict__ q_hit, float4* __restrict__ nq_o,
                float4* __restrict__ nq_d, float4* __restrict__ s_o, float4* __restrict__ s_d,
                float4* __restrict__ s_c, float4* __restrict__ weight, float4* __restrict__ rad, Counters* c,
                XcdQueue queue, NrcShade nrc, uint32_t omask) {
    pt_shade<false, Seed>(S, cur, bounce, max_depth, rr, q_o, q_d, q_hit, nq_o, nq_d, s_o, s_d, s_c, weight, rad, c,
                          queue, nrc, omask);
}

// Shade with the radiance cache: queries and training rows (NrcShade)
template <class Seed>
__global__ __launch_bounds__(kPtBlock)
void k_pt_shade_nrc(DevScene S, int cur, uint32_t bounce, uint32_t max_depth, int rr, const float4* __restrict__ q_o,
                    const float4* __restrict__ q_d, const float2* __restrict__ q_hit, float4* __restrict__ nq_o,
                    float4* __restrict__ nq_d, float4* __restrict__ s_o, float4* __restrict__ s_d,
                    float4* __restrict__ s_c, float4* __restrict__ weight, float4* __restrict__ rad, Counters* c,
                    XcdQueue queue, NrcShade nrc, uint32_t omask) {
    pt_shade<true, Seed>(S, cur, bounce, max_depth, rr, q_o, q_d, q_hit, nq_o, nq_d, s_o, s_d, s_c, weight, rad, c,
                         queue, nrc, omask);
}

// query count after the second bounce's shade: the queries inferred on the side stream
__global__ void k_snapshot_queries(Counters* c) { c->query_early.v = c->cache.queries; }

// training rows from the pending rows of finished training paths: target = (final radiance -
// radiance before the vertex's reflection) / throughput at the vertex (0 where the throughput is 0);
// also counts the batch's queries and rows. part_rows: whole paths leave their rows in parts of so many, one per XCD
// (0: in one list).
__device__ __forceinline__ void nrc_rows(uint32_t first, uint32_t stride, const float4* __restrict__ pending, Counters* c,
                                         uint32_t max_rows, uint32_t part_rows, const float4* __restrict__ rad,
                                         float4* __restrict__ rows) {
    uint32_t part[8], total = 0, queries = 0;
    if (part_rows != 0u) {
#pragma unroll
        for (uint32_t x = 0; x < 8; ++x) {
            part[x] = min(c->cache_part[x].rows, part_rows);
            total += part[x];
            queries += c->cache_part[x].queries;
        }
    } else {
        total = c->cache.rows;
        queries = c->cache.queries;
    }
    const uint32_t n = min(total, max_rows);
    if (part_rows != 0u && total > n) {  // too many: as large a share of every part, its first rows
        uint32_t before = 0, kept = 0;
#pragma unroll
        for (uint32_t x = 0; x < 8; ++x) {
            before += part[x];
            const uint32_t upto = (uint32_t)((unsigned long long)before * n / total);
            part[x] = upto - kept;
            kept = upto;
        }
    }
    if (first == 0) {
        c->cache_queries += queries;
        c->cache_rows += n;
        if (part_rows != 0u) c->cache.rows = total;  // for the training steps
    }
    for (uint32_t i = first; i < n; i += stride) {
        uint32_t slot = i;
        if (part_rows != 0u) {
            uint32_t left = i;
            bool found = false;
#pragma unroll
            for (uint32_t x = 0; x < 8; ++x) {
                if (!found && left < part[x]) {
                    slot = x * part_rows + left;
                    found = true;
                }
                left -= found ? 0u : part[x];
            }
        }
        const float4* r = pending + (size_t)slot * 6;
        const float4 a = r[4], b = r[5];
        const uint32_t p = __float_as_uint(b.z);
        const float4 R = rad[p];
        const float beta[3] = {a.w, b.x, b.y}, snap[3] = {a.x, a.y, a.z}, fin[3] = {R.x, R.y, R.z};
        float tgt[3];
        for (int k = 0; k < 3; ++k) tgt[k] = beta[k] > 0.0f ? (fin[k] - snap[k]) / beta[k] : 0.0f;
        float4* o = rows + (size_t)i * 5;
        for (int k = 0; k < 4; ++k) o[k] = r[k];
        o[4] = make_float4(tgt[0], tgt[1], tgt[2], 0.0f);
    }
}

// shadow ray i: visible -> radiance of its path += contribution (traceVisibility, :66-73)
__device__ __forceinline__ void shadow_result(bool occluded, const float4 d4, const float4* __restrict__ s_c,
                                              uint32_t i, float4* __restrict__ rad) {
    if (occluded) return;
    const uint32_t p = __float_as_uint(d4.w);
    const float4 cc = s_c[i];
    const float4 R = rad[p];
    v3 L = mk(R.x, R.y, R.z);
    L += mk(cc.x, cc.y, cc.z);
    rad[p] = make_float4(L.x, L.y, L.z, R.w);
}

// A wave's share of its XCD's len rays of one queue. They go to the XCD's waves in pieces: a wave's first
// piece is dealt by its index, the next ones come from the XCD's counter.
// What bounds the handing out is the counters: one 128-byte line serves an add with a return value
// every 13 ns when only its own XCD uses it, and other XCDs' reads in between hold every add up. With
// one add per refill of some 40 rays, the 20 M rays of a Cornell box bounce were 0.85 ms of counting
// in a launch of 1.76 ms; with waves that tried all 8 counters before they ended, a launch took at
// least 115 us however few rays it had, and one that refilled some 300 us. Hence the XCD's own counter
// only (the XCDs' shares of a queue are equal enough), and pieces of 64 to 256 rays: as many as leave
// each of the XCD's waves two more, so that they shrink towards the end. Gradient domain (Cornell box,
// 512x512, 16 spp) 9.5 -> 7.4 ms, volume renderer (512x512, 16 spp) 3.85 -> 2.63 ms, 1080p / 1M triangles /
// 64 spp 113.5 -> 109.8 ms. Pieces of up to 64, 512 and 1024 rays: 3% slower, the same, the same.
struct RayShare {
    XcdQueue queue;
    CounterLine* counter;    // the XCD's
    uint32_t waves;          // its number of waves
    uint32_t len, dealt;     // its rays, and those of the first pieces
    uint32_t at, end;        // the wave's piece
    __device__ __forceinline__ uint32_t piece(uint32_t left) const {
        return min(max(left / (2u * waves) & ~63u, 64u), 256u);
    }
    __device__ __forceinline__ void begin(XcdQueue q, CounterLine* c, uint32_t n) {
        queue = q;
        counter = c;
        waves = (gridDim.x >> 3) * kPtWaves;
        len = n;
        const uint32_t size = piece(len);
        dealt = min(size * waves, len);
        at = __builtin_amdgcn_readfirstlane(min(((blockIdx.x >> 3) * kPtWaves + (threadIdx.x >> 6)) * size, len));
        end = min(at + size, len);
    }
    // a new piece; false when there is none (wave-uniform: the whole wave calls it)
    __device__ __forceinline__ bool refill() {
        if (dealt == len) return false;
        const uint32_t size = piece(len - end);
        uint32_t base = 0;
        if (__lane_id() == 0u) base = atomicAdd(&counter->v, size);
        at = __builtin_amdgcn_readfirstlane(base) + dealt;
        end = min(at + size, len);
        return at < len;
    }
    __device__ __forceinline__ uint32_t index(uint32_t k) const { return queue.slot(blockIdx.x & 7u, k); }
};

// An XCD's n rays of one queue, dealt out by RayShare; finish(i, hit, r) consumes the result of the ray in slot i.
template <bool kAny, class Load, class Finish>
__device__ __forceinline__ void trace_queue(const DevScene& S, XcdQueue queue, uint32_t n, CounterLine* counter,
                                            LaneStack<kPtLds>& st, Load load, Finish finish) {
    RayShare share;
    share.begin(queue, counter, n);
    trace_pool<kAny, true>(S, share, st, load, finish);
}

// One bounce's extension rays (queue cur), then the previous bounce's shadow rays (parity cur ^ 1),
// each queue handed out by one counter per XCD (trace_queue; short launches and the visit-counting
// instantiation deal out 64-ray chunks instead, one ray per lane until the chunk is done).
// amdgpu_waves_per_eu(8, 8): the compiler keeps the kernel within the SGPR budget of 8 waves per
// SIMD (spilling a few SGPRs into VGPR lanes); without it 104 SGPRs held the kernel to 6 resident
// waves per SIMD and a quarter of the persistent blocks only started when the queue was empty.
template <bool kCount>
__global__ __launch_bounds__(kPtBlock) __attribute__((amdgpu_waves_per_eu(8, 8)))
void k_pt_trace(DevScene S, int cur, const float4* __restrict__ q_o, const float4* __restrict__ q_d,
                float2* __restrict__ q_hit, const float4* __restrict__ s_o, const float4* __restrict__ s_d,
                const float4* __restrict__ s_c, float4* __restrict__ rad, Counters* c, XcdQueue queue, uint32_t* spill,
                uint32_t spill_stride) {
    __shared__ uint32_t lds[kPtLds * kPtBlock];
    const uint32_t gtid = blockIdx.x * blockDim.x + threadIdx.x;
    // Workgroups are dispatched to the 8 XCDs round-robin: block b runs on XCD b % 8 (only the speed
    // depends on it) and traces that XCD's share of the queues
    const uint32_t xcd = blockIdx.x & 7u;
    const uint32_t n_ext = c->rays[cur ^ 1][xcd].ext, n_sh = c->rays[cur ^ 1][xcd].shadow;
    if (gtid < 8) {
        c->rays[cur][gtid].both = 0;
        c->inside[cur][gtid].v = 0;
        atomicAdd(&c->extension_rays, (unsigned long long)c->rays[cur ^ 1][gtid].ext);
        atomicAdd(&c->shadow_rays, (unsigned long long)c->rays[cur ^ 1][gtid].shadow);
    }
    LaneStack<kPtLds> st{lds + threadIdx.x, kPtBlock, spill ? spill + gtid : nullptr, spill_stride};
    TravCount te, ts;
    // the same decision for every wave of the XCD (n_ext and n_sh are read at the start)
    const bool refill = !kCount && n_ext + n_sh >= CUPBR_REFILL_MIN * (gridDim.x >> 3) * kPtBlock;
    if (refill && gtid == 0) c->refill_launches += 1;
    if (refill) {
        trace_queue<false>(
            S, queue, n_ext, &c->work[xcd], st,
            [&](uint32_t i, v3& o, v3& d, float& dist) {
                const float4 o4 = q_o[i], d4 = q_d[i];
                o = mk(o4.x, o4.y, o4.z);
                d = mk(d4.x, d4.y, d4.z);
                dist = 0.0f;
            },
            [&](uint32_t i, bool, const TraceResult& r) { q_hit[i] = make_float2(r.t, __uint_as_float(r.prim)); });
        trace_queue<true>(
            S, queue, n_sh, &c->swork[xcd], st,
            [&](uint32_t j, v3& o, v3& d, float& dist) {
                const float4 o4 = s_o[j], d4 = s_d[j];
                o = mk(o4.x, o4.y, o4.z);
                d = mk(d4.x, d4.y, d4.z);
                dist = o4.w;
            },
            [&](uint32_t j, bool occluded, const TraceResult&) { shadow_result(occluded, s_d[j], s_c, j, rad); });
    } else {
        // 64-ray chunks, one ray per lane until the chunk is done (and the visit-counting pass). The
        // XCD's chunks, extension then shadow, go to its waves one after the other. No counters: a wave
        // has one chunk (in the visit-counting pass as many as it takes). Cornell box, 256x256, 1 spp:
        // 730 -> 238 us a frame. Chunks of 32, 16 or 8 rays on more waves gave 247, 249 and 256 us.
        const uint32_t e_chunks = (n_ext + 63u) >> 6, chunks = e_chunks + ((n_sh + 63u) >> 6);
        const uint32_t waves = (gridDim.x >> 3) * kPtWaves;
        for (uint32_t q = (blockIdx.x >> 3) * kPtWaves + (threadIdx.x >> 6); q < chunks; q += waves) {
            if (q < e_chunks) {
                const uint32_t r = (q << 6) + __lane_id(), i = queue.slot(xcd, r);
                if (r < n_ext) {
                    const float4 o4 = q_o[i], d4 = q_d[i];
                    TraceResult hit;
                    traverse<false, kPtLds, kCount>(S, mk(o4.x, o4.y, o4.z), mk(d4.x, d4.y, d4.z), 0.0f, st, hit, &te);
                    q_hit[i] = make_float2(hit.t, __uint_as_float(hit.prim));
                }
            } else {
                const uint32_t r = ((q - e_chunks) << 6) + __lane_id(), j = queue.slot(xcd, r);
                if (r < n_sh) {
                    const float4 o4 = s_o[j], d4 = s_d[j];
                    TraceResult hit;
                    const bool occluded = traverse<true, kPtLds, kCount>(S, mk(o4.x, o4.y, o4.z),
                                                                          mk(d4.x, d4.y, d4.z), o4.w, st, hit, &ts);
                    shadow_result(occluded, d4, s_c, j, rad);
                }
            }
        }
    }
    if (kCount) {
        wave_add_counts(te, &c->ext_nodes, &c->ext_prims);
        wave_add_counts(ts, &c->shadow_nodes, &c->shadow_prims);
    }
}

// Bounce 0 (PathTracer.cu:112-126): the camera rays, made where they are traced and traced as
// packets. Queue slot chunks of 64 (SampleOrder: the samples of one pixel, or of a few neighbouring
// pixels, or an 8x8 pixel tile; GDPT: the five paths of about 13 neighbouring pixels) hold rays that
// leave the camera position in nearby directions, so each wave runs traverse_packet over one chunk.
// Blocks are dispatched to the 8 XCDs round-robin; block b takes chunk range
// (b % 8) * (gridDim.x / 8) + b / 8, so each XCD traces a contiguous eighth of the queue
// (neighbouring tiles share its L2). gridDim.x is a multiple of 8; n = queue 0's length.
// make(i, o, d) makes slot i's ray and writes the path's state. Queue 0 holds one origin, in slot 0:
// every camera ray leaves the camera position, and the first shade reads it for all (omask = 0); in it a
// path's id is its slot, its throughput 1, and the generator state takes the id's place (a pass over the
// throughputs less in both kernels: 512x512, 16 spp, gradient domain 6.67 -> 6.57 ms).
template <class Make>
__device__ __forceinline__ void camera_packets(const DevScene& S, uint32_t n, float4* __restrict__ q_o,
                                               float2* __restrict__ q_hit, Make make) {
    const uint32_t blk = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    const uint32_t wave_first = blk * kPtBlock + (threadIdx.x & ~63u);
    if (wave_first >= n) return;  // whole waves only: traverse_packet needs all 64 lanes
    const uint32_t i = wave_first + __lane_id();
    const bool valid = i < n;
    v3 o = splat(0.0f), d = mk(0.0f, 0.0f, 1.0f);
    if (valid) make(i, o, d);
    if (i == 0u) q_o[0] = make_float4(o.x, o.y, o.z, 0.0f);
    TraceResult r;
    traverse_packet(S, o, d, valid, r);
    if (valid) q_hit[i] = make_float2(r.t, __uint_as_float(r.prim));
}

// bounce 0 of a path-tracer or volume-renderer batch: the rays of k_pt_raygen, traced at once;
// it also resets the batch's counters
template <class Seed>
__global__ __launch_bounds__(kPtBlock) __attribute__((amdgpu_waves_per_eu(8, 8)))
void k_pt_camera(DevScene S, uint32_t n, cupbr_camera cam, uint32_t w, uint32_t h, uint32_t frame0, SampleOrder order,
                 uint32_t train_thresh, float4* __restrict__ q_o, float4* __restrict__ q_d,
                 float4* __restrict__ rad, float2* __restrict__ q_hit, Counters* c,
                 XcdQueue queue) {
    if (blockIdx.x == 0 && threadIdx.x < 8) reset_batch_counters(c, queue, n, threadIdx.x);
    if (blockIdx.x == 0 && threadIdx.x == 0) c->extension_rays += n;
    camera_packets(S, n, q_o, q_hit, [&](uint32_t i, v3& o, v3& d) {
        Seed seed;
        uint32_t pix, frame;
        camera_path(cam, w, h, frame0, order, i, seed, pix, frame, o, d);
        q_d[i] = make_float4(d.x, d.y, d.z, __uint_as_float(state_bits(seed)));
        rad[i] = make_float4(0.0f, 0.0f, 0.0f, __uint_as_float(is_training_path(pix, frame, train_thresh) ? 1u : 0u));
    });
}

// Slots of two lists for the lanes of a wave that want one, whose counts are the halves of *counts: one add.
__device__ __forceinline__ void wave_append2(bool want_lo, bool want_hi, unsigned long long* counts, uint32_t& lo,
                                             uint32_t& hi) {
    const unsigned long long ml = __ballot(want_lo), mh = __ballot(want_hi), below = (1ull << __lane_id()) - 1ull;
    unsigned long long base = 0;
    if ((ml | mh) != 0ull && __lane_id() == 0u)
        base = atomicAdd(counts, (unsigned long long)__popcll(mh) << 32 | (unsigned long long)__popcll(ml));
    lo = __builtin_amdgcn_readfirstlane((uint32_t)base) + (uint32_t)__popcll(ml & below);
    hi = __builtin_amdgcn_readfirstlane((uint32_t)(base >> 32)) + (uint32_t)__popcll(mh & below);
}

// paths of one XCD in a k_pt_paths launch of so many blocks
__host__ __device__ inline uint32_t part_paths(uint32_t blocks, uint32_t per_wave) { return (blocks >> 3) * kPtWaves * per_wave; }

// Whole paths of a small batch: the camera rays as packets (camera_packets), then vertex, shadow ray and next ray in
// turn, in the order of the kernels above, so that a path's radiance is the same sum. per_wave paths a wave; with
// kFew its last 16 and fewer rays by 8 lanes each (trace_lanes). nrc.max_rows: pending rows of one XCD's part.
template <bool kNrc, bool kFew, class Seed>
__global__ __launch_bounds__(kPtBlock)
void k_pt_paths(DevScene S, uint32_t n, uint32_t per_wave, cupbr_camera cam, uint32_t w, uint32_t h, uint32_t frame0,
                SampleOrder order, uint32_t train_thresh, uint32_t max_depth, int rr, float4* __restrict__ rad,
                Counters* c, NrcShade nrc, uint32_t* spill, uint32_t spill_stride) {
    __shared__ uint32_t lds[kPtLds * kPtBlock];
    const uint32_t gtid = blockIdx.x * blockDim.x + threadIdx.x;
    LaneStack<kPtLds> st{lds + threadIdx.x, kPtBlock, spill ? spill + gtid : nullptr, spill_stride};
    const uint32_t blk = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    const uint32_t wave_first = (blk * kPtWaves + (threadIdx.x >> 6)) * per_wave;
    if (wave_first >= n) return;  // whole waves only: traverse_packet needs all 64 lanes
    const uint32_t p = wave_first + __lane_id();
    const bool mine = __lane_id() < per_wave && p < n;
    bool alive = mine;
    v3 o = splat(0.0f), d = mk(0.0f, 0.0f, 1.0f), w3 = splat(1.0f), L = splat(0.0f);
    Seed seed{};
    bool training = false;
    if (alive) {
        uint32_t pix, frame;
        camera_path(cam, w, h, frame0, order, p, seed, pix, frame, o, d);
        training = is_training_path(pix, frame, train_thresh);
    }
    TraceResult r;
    traverse_packet(S, o, d, alive, r);
    uint32_t n_ext = alive ? 1u : 0u, n_sh = 0;
    // an XCD's cache records go to its own part of the lists (a path asks the cache once, so its queries fit the range
    // of its paths). With one counter that all XCDs add to at each bounce this kernel takes, in the Cornell box with
    // training, 97 instead of 89 us (256x256) and 194 instead of 170 (300x299, 2 spp); with a frozen cache, whose paths
    // ask once, 106 instead of 110.
    const uint32_t xcd = blockIdx.x & 7u;
    unsigned long long* const counts = &c->cache_part[xcd].both;
    float4* const queries = nrc.queries + (size_t)xcd * part_paths(gridDim.x, per_wave) * 5u;
    float4* const pending = nrc.pending + (size_t)xcd * nrc.max_rows * 6u;
    for (uint32_t bounce = 0;; ++bounce) {
        Vertex v;
        v.next = v.shadow = v.query = v.row = false;
        if (alive) {
            path_vertex<kNrc, Seed>(S, bounce, max_depth, rr, nrc, o, d, r.t, r.prim, p, training, L, w3, seed, v);
            if (v.emits) L += v.emission;
        }
        if (kNrc) {
            uint32_t qs, rs;
            wave_append2(v.query, v.row, counts, qs, rs);
            if (v.query)
                for (int k = 0; k < 5; ++k) queries[qs * 5u + k] = v.rec[k];
            if (v.row && rs < nrc.max_rows)
                for (int k = 0; k < 6; ++k) pending[rs * 6u + k] = v.rec[k];
        }
        bool occluded = false;
        n_sh += v.shadow ? 1u : 0u;
        if (kFew)
            occluded = trace_lanes<true>(S, v.shadow, v.shadow_o, v.shadow_d, v.dist, st, r);
        else if (v.shadow)
            occluded = traverse<true>(S, v.shadow_o, v.shadow_d, v.dist, st, r);
        if (v.shadow && !occluded) L += v.light;
        alive = v.next;
        if (__ballot(alive) == 0ull) break;
        n_ext += alive ? 1u : 0u;
        o = v.next_o;
        d = v.next_d;
        if (kFew)
            trace_lanes<false>(S, alive, o, d, 0.0f, st, r);
        else if (alive)
            traverse<false>(S, o, d, 0.0f, st, r);
    }
    if (mine) rad[p] = make_float4(L.x, L.y, L.z, __uint_as_float(training ? 1u : 0u));
    for (int off = 32; off > 0; off >>= 1) {
        n_ext += __shfl_xor(n_ext, off);
        n_sh += __shfl_xor(n_sh, off);
    }
    if (__lane_id() == 0u) {
        atomicAdd(&c->extension_rays, (unsigned long long)n_ext);
        atomicAdd(&c->shadow_rays, (unsigned long long)n_sh);
    }
}

// The running mean of PathTracer.cu:162-168 per pixel, frame by frame in order. A pixel's samples
// are runs of consecutive slots (SampleOrder: up to f frames); a thread loads up to 8 of them at
// once, so that the 128-byte line they share is fetched once.
__device__ __forceinline__ void accumulate_pixel(uint32_t pix, float* __restrict__ img, const float4* __restrict__ rad,
                                                 uint32_t w, uint32_t h, SampleOrder order, uint32_t frame0,
                                                 uint32_t nspp) {
    if (pix >= w * h) return;
    const uint32_t py = pix / w, j = tile_slot(pix - py * w, py, w, h);
    v3 acc = ld3(img + 3 * (size_t)pix);
    for (uint32_t s = 0; s < nspp;) {
        const uint32_t base = order.slot(s, j);
        const uint32_t run = min(order.f - s % order.f, nspp - s);  // slots base .. base + run - 1
        for (uint32_t k = 0; k < run; k += 8) {
            const uint32_t m = min(8u, run - k);
            float4 R[8];
#pragma unroll
            for (uint32_t q = 0; q < 8; ++q)
                if (q < m) R[q] = rad[base + k + q];
#pragma unroll
            for (uint32_t q = 0; q < 8; ++q) {
                if (q >= m) break;
                const v3 L = mk(R[q].x, R[q].y, R[q].z);
                const uint32_t f = frame0 + s + k + q;
                if (f > 0) {
                    const float a = 1.0f / ((float)f + 1.0f);
                    acc = (1.0f - a) * acc + a * L;
                } else {
                    acc = L;
                }
            }
        }
        s += run;
    }
    st3(img + 3 * (size_t)pix, acc);
}

__global__ __launch_bounds__(kPtBlock) void k_accumulate(float* __restrict__ img, const float4* __restrict__ rad,
                                                         uint32_t w, uint32_t h, SampleOrder order, uint32_t frame0,
                                                         uint32_t nspp) {
    accumulate_pixel(blockIdx.x * blockDim.x + threadIdx.x, img, rad, w, h, order, frame0, nspp);
}

// the same with the radiance cache, and the batch's training rows (nrc_rows) in the blocks from pix_blocks on
__global__ __launch_bounds__(kPtBlock) void k_accumulate_rows(float* __restrict__ img, const float4* __restrict__ rad,
                                                              uint32_t w, uint32_t h, SampleOrder order, uint32_t frame0,
                                                              uint32_t nspp, uint32_t pix_blocks,
                                                              const float4* __restrict__ pending, Counters* c,
                                                              uint32_t max_rows, uint32_t part_rows,
                                                              float4* __restrict__ rows) {
    if (blockIdx.x < pix_blocks)
        accumulate_pixel(blockIdx.x * blockDim.x + threadIdx.x, img, rad, w, h, order, frame0, nspp);
    else
        nrc_rows((blockIdx.x - pix_blocks) * blockDim.x + threadIdx.x, (gridDim.x - pix_blocks) * blockDim.x, pending, c,
                 max_rows, part_rows, rad, rows);
}

// ------------------------------------------------------------------ gradient-domain paths
// gdpt_kernel (GradientDomain.cu:160-246) on the same queues. A group is one interior pixel of one
// frame: its base path and four shifted paths (left, right, up, down), path ids 5g + k. Each
// follows collect_radiance (:110-158) on its own part of the group's seed chain; a shifted path
// stops at the first depth where the base path has no vertex (:126-127). All five advance bounce
// by bounce: the base path's shade of bounce b records the queue slot of its bounce-(b+1) ray (or
// none) in slot[(b+1) & 1][g], and a shifted path's shade of bounce b+1 reads that ray's hit, one
// launch later. A shifted path alive at bounce b passed the check at b-1, so the base path was
// shaded at b-1 and wrote the slot it reads: no stale entries, no reads of what the same launch
// writes. Queue slots of a frame's groups follow the 8x8 tiles of the interior pixels.
constexpr uint32_t kNoSlot = 0xFFFFFFFFu;

// The camera ray of GDPT path pid = 5 g + k (g = frame s of interior pixel gi; k: base, left,
// right, up, down), and its generator state after the ray's draws (GradientDomain.cu:180-213).
__device__ __forceinline__ void gdpt_camera_path(const cupbr_camera& cam, uint32_t w, uint32_t h, uint32_t frame0,
                                                 uint32_t n_int, uint32_t pid, uint32_t& chain, v3& o, v3& d) {
    const uint32_t g = pid / 5u, k = pid - 5u * g;
    const uint32_t s = g / n_int, gi = g - s * n_int;
    uint32_t ix, iy;
    tile_pixel(gi, w - 2u, h - 2u, ix, iy);
    const uint32_t px = ix + 1u, py = iy + 1u;
    // the five camera rays of a group come from one chain, base, left, right, up, down, two draws
    // each; each path continues from the chain as it stood after its own ray (:180-213). Path k
    // skips the 2k draws of the rays before its own.
    chain = tea4(py * w + px, frame0 + s);
    for (uint32_t j = 0; j < 2u * k; ++j) chain = 1664525u * chain + 1013904223u;  // rnd's state step
    const uint32_t nx = k == 1 ? px - 1u : (k == 2 ? px + 1u : px);
    const uint32_t ny = k == 3 ? py + 1u : (k == 4 ? py - 1u : py);
    launch_ray(nx, ny, w, h, cam, chain, o, d);
}

__global__ __launch_bounds__(kPtBlock) void k_gdpt_raygen(cupbr_camera cam, uint32_t w, uint32_t h, uint32_t frame0,
                                                          uint32_t n_int, uint32_t n_groups, float4* __restrict__ q_o,
                                                          float4* __restrict__ q_d, float4* __restrict__ weight,
                                                          float4* __restrict__ rad, uint32_t* __restrict__ slot0,
                                                          Counters* c, XcdQueue queue) {
    // one thread per path, so that the queue and state writes of a wave are contiguous
    const uint32_t pid = blockIdx.x * blockDim.x + threadIdx.x;
    if (pid < 8) reset_batch_counters(c, queue, 5u * n_groups, pid);
    if (pid >= 5u * n_groups) return;
    uint32_t chain;
    v3 o, d;
    gdpt_camera_path(cam, w, h, frame0, n_int, pid, chain, o, d);
    q_o[pid] = make_float4(o.x, o.y, o.z, 0.0f);
    q_d[pid] = make_float4(d.x, d.y, d.z, __uint_as_float(pid));
    weight[pid] = make_float4(1.0f, 1.0f, 1.0f, __uint_as_float(chain));
    rad[pid] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (pid % 5u == 0u) slot0[pid / 5u] = pid;
}

// bounce 0 of a GDPT batch: the rays of k_gdpt_raygen, traced at once (camera_packets); it also
// resets the batch's counters. n = 5 x the batch's groups.
__global__ __launch_bounds__(kPtBlock) __attribute__((amdgpu_waves_per_eu(8, 8)))
void k_gdpt_camera(DevScene S, uint32_t n, cupbr_camera cam, uint32_t w, uint32_t h, uint32_t frame0, uint32_t n_int,
                   float4* __restrict__ q_o, float4* __restrict__ q_d,
                   float4* __restrict__ rad, uint32_t* __restrict__ slot0, float2* __restrict__ q_hit, Counters* c,
                   XcdQueue queue) {
    if (blockIdx.x == 0 && threadIdx.x < 8) reset_batch_counters(c, queue, n, threadIdx.x);
    if (blockIdx.x == 0 && threadIdx.x == 0) c->extension_rays += n;
    camera_packets(S, n, q_o, q_hit, [&](uint32_t i, v3& o, v3& d) {
        uint32_t chain;
        gdpt_camera_path(cam, w, h, frame0, n_int, i, chain, o, d);
        q_d[i] = make_float4(d.x, d.y, d.z, __uint_as_float(chain));
        rad[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (i % 5u == 0u) slot0[i / 5u] = i;
    });
}

// one bounce of collect_radiance (:121-156) for every queued path. amdgpu_waves_per_eu(4, 8): 95 VGPRs and 5 waves
// per SIMD since it touches only the state that changes. (Before that, with 102 VGPRs at 4 waves, forcing 5 waves
// cost 1.6%, and 6 waves, with a 24-byte spill, 5%: Cornell box 512², 128 spp, 504, 496 and 478 Msamples/s.)
__global__ __launch_bounds__(kPtBlock) __attribute__((amdgpu_waves_per_eu(4, 8)))
void k_gdpt_shade(DevScene S, int cur, uint32_t bounce, uint32_t max_depth, const float4* __restrict__ q_o,
                  const float4* __restrict__ q_d, const float2* __restrict__ q_hit, float4* __restrict__ nq_o,
                  float4* __restrict__ nq_d, float4* __restrict__ s_o, float4* __restrict__ s_d,
                  float4* __restrict__ s_c, float4* __restrict__ weight, float4* __restrict__ rad, Counters* c,
                  XcdQueue queue, const uint32_t* __restrict__ slot_now, uint32_t* __restrict__ slot_next,
                  uint32_t omask) {
    __shared__ uint32_t s_append[2 * (kPtWaves + 1)];
    const uint32_t xcd = blockIdx.x & 7u, n = c->rays[cur ^ 1][xcd].ext;
    if (blockIdx.x == 0 && threadIdx.x < 8) c->work[threadIdx.x].v = c->swork[threadIdx.x].v = 0;
    const float nl = (float)(S.n_lights + (S.use_env ? 1u : 0u));
    for (uint32_t base = (blockIdx.x >> 3) * kPtBlock; base < n; base += (gridDim.x >> 3) * kPtBlock) {
        const uint32_t i = queue.slot(xcd, base + threadIdx.x);
        bool want_next = false, want_shadow = false;
        float4 no = {}, nd = {}, so = {}, sd = {}, sc = {};
        if (base + threadIdx.x < n) {
            const float4 o4 = q_o[i & omask], d4 = q_d[i];
            const float2 hh = q_hit[i];
            const bool first = omask == 0u;
            const uint32_t p = first ? i : __float_as_uint(d4.w);
            const uint32_t g = p / 5u, k = p - 5u * g;
            bool go = true;
            if (k != 0) {  // :126-127: the base path needs a vertex at this depth
                const uint32_t bs = slot_now[g];
                go = bs != kNoSlot && __float_as_uint(q_hit[bs].y) != kNoHit;
            }
            if (go) {
                const float4 W = first ? make_float4(1.0f, 1.0f, 1.0f, d4.w) : weight[p];
                v3 w3 = mk(W.x, W.y, W.z);
                uint32_t seed = __float_as_uint(W.w);
                // most vertices add none, and their radiance is neither read nor written; a throughput is written for
                // paths that go on (512x512, 16 spp: 6.95 -> 6.67 ms; volume renderer 2.58 -> 2.53)
                v3 emission = splat(0.0f);
                const v3 o = mk(o4.x, o4.y, o4.z), d = mk(d4.x, d4.y, d4.z);
                const uint32_t prim = __float_as_uint(hh.y);
                if (prim == kNoHit) {  // :128-137
                    if (S.use_env) emission = w3 * env_lookup(S, d);
                } else {
                    const v3 P = o + hh.x * d;
                    v3 N;
                    uint32_t obj;
                    hit_geometry(S, prim, P, N, obj);
                    const Mat m = load_mat(S.mats + obj);
                    const v3 inc = -1.0f * d;
                    emission = w3 * m.albedo_e;  // emissiveIllumintationGDPT :39-44
                    if (m.type != CUPBR_GLASS && dot(N, inc) <= 0.0f) {  // directIlluminationGDPT :46-88
                        w3 = splat(0.0f);
                    } else {
                        v3 ldir, le;
                        float dist = 0.0f;
                        if (nee_sample(S, m, seed, P, inc, N, ldir, le, dist)) {
                            const v3 contrib = (nl * fmaxf(0.0f, dot(N, ldir))) * brdf(m, inc, ldir, N) * le * w3;
                            if (!(contrib.x == 0.0f && contrib.y == 0.0f && contrib.z == 0.0f)) {
                                const v3 sorg = P + 0.001f * ldir;
                                const v3 sdir = normalize(ldir);
                                want_shadow = true;
                                so = make_float4(sorg.x, sorg.y, sorg.z, dist);
                                sd = make_float4(sdir.x, sdir.y, sdir.z, __uint_as_float(p));
                                sc = make_float4(contrib.x, contrib.y, contrib.z, 0.0f);
                            }
                        }
                    }
                    // indirectIlluminationGDPT :90-108 (a zero weight keeps the path going: the
                    // base path's later vertices decide how far its shifted paths go)
                    const DirPdf sp = sample_direction(m, seed, inc, N);
                    if (!(norm(sp.d) == 0.0f)) {
                        w3 = w3 * fabsf(dot(sp.d, N)) * brdf(m, inc, sp.d, N) / sp.pdf;
                        if (bounce + 1 < max_depth) {  // :154-156
                            const v3 norg = P + 0.01f * sp.d;
                            const v3 ndir = normalize(sp.d);
                            want_next = true;
                            no = make_float4(norg.x, norg.y, norg.z, 0.0f);
                            nd = make_float4(ndir.x, ndir.y, ndir.z, __uint_as_float(p));
                        }
                    }
                    if (want_next) weight[p] = make_float4(w3.x, w3.y, w3.z, __uint_as_float(seed));
                }
                if (!(emission.x == 0.0f && emission.y == 0.0f && emission.z == 0.0f)) {
                    const float4 R = rad[p];
                    rad[p] = make_float4(R.x + emission.x, R.y + emission.y, R.z + emission.z, R.w);
                }
            }
            if (k == 0) slot_next[g] = kNoSlot;  // overwritten below when the base path goes on
        }
        uint32_t ns, ss;
        block_append2(want_next, want_shadow, &c->rays[cur][xcd].both, s_append, ns, ss);
        if (want_next) {
            ns = queue.slot(xcd, ns);
            nq_o[ns] = no;
            nq_d[ns] = nd;
            const uint32_t p = __float_as_uint(nd.w);
            const uint32_t g = p / 5u;
            if (p == 5u * g) slot_next[g] = ns;
        }
        if (want_shadow) {
            ss = queue.slot(xcd, ss);
            s_o[ss] = so;
            s_d[ss] = sd;
            s_c[ss] = sc;
        }
    }
}

// gradients and running means of the five buffers (:214-245), frame by frame in order
__global__ __launch_bounds__(kPtBlock) void k_gdpt_accumulate(float* __restrict__ base, float* __restrict__ gxf,
                                                              float* __restrict__ gxb, float* __restrict__ gyf,
                                                              float* __restrict__ gyb, const float4* __restrict__ rad,
                                                              uint32_t w, uint32_t h, uint32_t n_int, uint32_t frame0,
                                                              uint32_t nspp) {
    const uint32_t gi = blockIdx.x * blockDim.x + threadIdx.x;
    if (gi >= n_int) return;
    uint32_t ix, iy;
    tile_pixel(gi, w - 2u, h - 2u, ix, iy);
    const size_t i3 = 3 * ((size_t)(iy + 1u) * w + ix + 1u);
    v3 acc[5] = {ld3(base + i3), ld3(gxf + i3), ld3(gxb + i3), ld3(gyf + i3), ld3(gyb + i3)};
    for (uint32_t s = 0; s < nspp; ++s) {
        const size_t p = 5 * ((size_t)s * n_int + gi);
        v3 L[5];
        for (int k = 0; k < 5; ++k) {
            const float4 R = rad[p + k];
            L[k] = mk(R.x, R.y, R.z);
        }
        const v3 val[5] = {L[0], 0.5f * (L[0] - L[1]), 0.5f * (L[2] - L[0]), 0.5f * (L[0] - L[4]),
                           0.5f * (L[3] - L[0])};
        const uint32_t f = frame0 + s;
        for (int k = 0; k < 5; ++k) {
            if (f > 0) {
                const float a = 1.0f / ((float)f + 1.0f);
                acc[k] = (1.0f - a) * acc[k] + a * val[k];
            } else {
                acc[k] = val[k];
            }
        }
    }
    st3(base + i3, acc[0]);
    st3(gxf + i3, acc[1]);
    st3(gxb + i3, acc[2]);
    st3(gyf + i3, acc[3]);
    st3(gyb + i3, acc[4]);
}

// ------------------------------------------------------------------ volume renderer paths
// volume_kernel (VolumeRenderer.cu:214-310) on the same queues, one iteration of its loop per
// bounce. A path's medium state lives in rad[p].w: bit 31 = inside an object, bits 0..30 = that
// object (the last interface crossed). Rays outside are traced by the trace kernels against the
// scene; rays inside go to the inside queue and are traced by the shade kernel against their
// object alone (Tracing::traceRay(scene, ray, index), TracingDetail.h:68-116), whose primitives it
// loops over. A path whose weight becomes zero (absorbed, back-facing, Russian roulette) stops:
// every later term would be multiplied by that weight.
constexpr uint32_t kInsideBit = 0x80000000u;

__global__ __launch_bounds__(kPtBlock) __attribute__((amdgpu_waves_per_eu(4, 8)))
void k_vol_shade(DevScene S, int cur, uint32_t bounce, uint32_t max_depth, int rr, const float4* __restrict__ q_o,
                 const float4* __restrict__ q_d, const float2* __restrict__ q_hit, const float4* __restrict__ iq_o,
                 const float4* __restrict__ iq_d, float4* __restrict__ nq_o, float4* __restrict__ nq_d,
                 float4* __restrict__ niq_o, float4* __restrict__ niq_d, float4* __restrict__ s_o,
                 float4* __restrict__ s_d, float4* __restrict__ s_c, float4* __restrict__ weight,
                 float4* __restrict__ rad, Counters* c, XcdQueue queue, uint32_t omask) {
    __shared__ uint32_t s_append[2 * (kPtWaves + 1)];
    const uint32_t xcd = blockIdx.x & 7u;
    const uint32_t n_out = c->rays[cur ^ 1][xcd].ext, n_in = c->inside[cur ^ 1][xcd].v, n = n_out + n_in;
    if (blockIdx.x == 0 && threadIdx.x < 8) c->work[threadIdx.x].v = c->swork[threadIdx.x].v = 0;
    const float nl = (float)(S.n_lights + (S.use_env ? 1u : 0u));
    unsigned long long inside_traces = 0;
    for (uint32_t base = (blockIdx.x >> 3) * kPtBlock; base < n; base += (gridDim.x >> 3) * kPtBlock) {
        const uint32_t r = base + threadIdx.x;
        const bool from_inside = r >= n_out;
        const uint32_t i = queue.slot(xcd, from_inside ? r - n_out : r);
        bool want_next = false, want_shadow = false, next_inside = false;
        float4 no = {}, nd = {}, so = {}, sd = {}, sc = {};
        if (r < n) {
            const float4 o4 = from_inside ? iq_o[i] : q_o[i & omask];
            const float4 d4 = from_inside ? iq_d[i] : q_d[i];
            const bool first = omask == 0u;
            const uint32_t p = first ? i : __float_as_uint(d4.w);
            const float4 W = first ? make_float4(1.0f, 1.0f, 1.0f, d4.w) : weight[p];
            const float4 R = rad[p];
            v3 w3 = mk(W.x, W.y, W.z);
            uint32_t seed = __float_as_uint(W.w);
            v3 emission = splat(0.0f);
            const uint32_t vstate = __float_as_uint(R.w);
            bool inside = (vstate & kInsideBit) != 0u;
            uint32_t obj_index = vstate & ~kInsideBit;
            const v3 o = mk(o4.x, o4.y, o4.z), d = mk(d4.x, d4.y, d4.z);
            TraceResult hr;
            if (from_inside) {
                ++inside_traces;
                object_trace(S, obj_index, o, d, hr);
            } else {
                const float2 hh = q_hit[i];
                hr.t = hh.x;
                hr.prim = __float_as_uint(hh.y);
            }
            const v3 inc = -1.0f * d;
            if (hr.prim == kNoHit) {  // :253-260
                if (S.use_env) emission = w3 * env_lookup(S, d);
            } else {
                const v3 P = o + hr.t * d;
                v3 N;
                uint32_t obj;
                hit_geometry(S, hr.prim, P, N, obj);
                const Mat m = load_mat(S.mats + obj);
                const int32_t vol_obj = inside ? (int32_t)obj : -1;  // the payload's volume (:277)
                bool next_valid = false, alive = true, medium_event = false;
                v3 out_dir = splat(0.0f), ray_start = splat(0.0f);
                // handleMediumInteraction :88-212
                const VolCoef vc = vol_coef(S, vol_obj);
                const v3 st = vc.sa + vc.ss;
                uint32_t ch = (uint32_t)(rnd(seed) * 3.0f);
                ch = min(ch, 2u);
                const float stc = comp(st, (int)ch);
                if (!safe_float_equal(stc, 0.0f)) {
                    const float t = -logf(1.0f - rnd(seed)) / stc;
                    if (t < hr.t) {
                        medium_event = true;
                        const v3 ep = o + t * d;
                        const float sprob = comp(vc.ss, (int)ch) / stc;
                        if (rnd(seed) < sprob) {
                            float pdf = 0.0f;
                            for (int k = 0; k < 3; ++k) pdf += comp(st, k) * expf(-1.0f * comp(st, k) * t);
                            pdf /= 3.0f;
                            w3 = w3 * vc.ss / sprob * vexp(-1.0f * st * t) / pdf;
                            v3 ldir, le;
                            float dist;
                            if (nee_sample(S, m, seed, ep, inc, N, ldir, le, dist)) {
                                const v3 sdir = normalize(ldir);
                                v3 sorg, att = splat(1.0f);
                                if (inside) {  // to the object's boundary first (:159-171)
                                    ++inside_traces;
                                    TraceResult ge;
                                    float gd = 0.0f;
                                    v3 gp = ep;
                                    if (object_trace(S, obj_index, ep, sdir, ge)) {
                                        gd = ge.t;
                                        gp = ep + ge.t * sdir;
                                    }
                                    att = vexp(-1.0f * st * gd) * hg_phase(vc.g, -dot(inc, ldir));
                                    sorg = gp + 0.001f * ldir;
                                    dist -= gd;
                                } else {
                                    sorg = ep + 0.001f * ldir;
                                }
                                const v3 sst = ld3(S.volume.sigma_a) + ld3(S.volume.sigma_s);
                                const v3 contrib = nl * vexp(-1.0f * sst * fminf(dist, 100000000.0f)) * att * le * w3;
                                if (!(contrib.x == 0.0f && contrib.y == 0.0f && contrib.z == 0.0f)) {
                                    want_shadow = true;
                                    so = make_float4(sorg.x, sorg.y, sorg.z, dist);
                                    sd = make_float4(sdir.x, sdir.y, sdir.z, __uint_as_float(p));
                                    sc = make_float4(contrib.x, contrib.y, contrib.z, 0.0f);
                                }
                            }
                            const DirPdf hs = hg_sample(vc.g, -1.0f * inc, seed);
                            out_dir = hs.d;
                            ray_start = ep;
                            next_valid = true;
                        } else {
                            alive = false;  // absorbed (:120-125)
                        }
                    } else {
                        float pdf = 0.0f;
                        for (int k = 0; k < 3; ++k) pdf += expf(-comp(st, k) * hr.t);
                        pdf /= 3.0f;
                        w3 = w3 * vexp(-1.0f * st * hr.t) / pdf;
                        ray_start = P;
                    }
                }
                if (alive && !medium_event) {
                    if (m.type == CUPBR_VOLUME_MATERIAL) {  // medium interface :269-278
                        const DirPdf sdp = sample_direction(m, seed, inc, N);
                        out_dir = sdp.d;
                        ray_start = P;
                        const bool refl = dot(inc, N) * dot(out_dir, N) > 0;
                        inside = refl ? inside : !inside;
                        obj_index = obj;
                        next_valid = true;
                    } else {
                        if (m.type != CUPBR_GLASS && dot(N, inc) <= 0.0f) {  // :24-70
                            w3 = splat(0.0f);
                        } else {
                            v3 ldir, le;
                            float dist;
                            if (nee_sample(S, m, seed, P, inc, N, ldir, le, dist)) {
                                const v3 contrib = (nl * fmaxf(0.0f, dot(N, ldir))) *
                                                   vexp(-1.0f * (vc.ss + vc.sa) * fminf(dist, 100000000.0f)) *
                                                   brdf(m, inc, ldir, N) * le * w3;
                                if (!(contrib.x == 0.0f && contrib.y == 0.0f && contrib.z == 0.0f)) {
                                    const v3 sorg = P + 0.001f * ldir;
                                    const v3 sdir = normalize(ldir);
                                    want_shadow = true;
                                    so = make_float4(sorg.x, sorg.y, sorg.z, dist);
                                    sd = make_float4(sdir.x, sdir.y, sdir.z, __uint_as_float(p));
                                    sc = make_float4(contrib.x, contrib.y, contrib.z, 0.0f);
                                }
                            }
                        }
                        const DirPdf sdp = sample_direction(m, seed, inc, N);  // :72-86
                        if (!(norm(sdp.d) == 0.0f)) {
                            w3 = w3 * fabsf(dot(sdp.d, N)) * brdf(m, inc, sdp.d, N) / sdp.pdf;
                            out_dir = sdp.d;
                            ray_start = P;
                            next_valid = true;
                        }
                    }
                    if (rr) {  // :280-289
                        const float alpha = clampf(fmaxf(w3.x, fmaxf(w3.y, w3.z)), 0.0f, 1.0f);
                        if (rnd(seed) > alpha || safe_float_equal(alpha, 0.0f)) {
                            next_valid = false;
                        } else {
                            w3 = w3 / alpha;
                        }
                    }
                }
                if (alive && next_valid && bounce + 1 < max_depth && !(w3.x == 0.0f && w3.y == 0.0f && w3.z == 0.0f)) {
                    const v3 norg = ray_start + 0.001f * out_dir;  // :298
                    const v3 ndir = normalize(out_dir);
                    want_next = true;
                    next_inside = inside;
                    no = make_float4(norg.x, norg.y, norg.z, 0.0f);
                    nd = make_float4(ndir.x, ndir.y, ndir.z, __uint_as_float(p));
                }
                if (want_next) weight[p] = make_float4(w3.x, w3.y, w3.z, __uint_as_float(seed));
            }
            const uint32_t state_now = (inside ? kInsideBit : 0u) | obj_index;
            if (state_now != vstate || !(emission.x == 0.0f && emission.y == 0.0f && emission.z == 0.0f))
                rad[p] = make_float4(R.x + emission.x, R.y + emission.y, R.z + emission.z, __uint_as_float(state_now));
        }
        const bool app_out = want_next && !next_inside, app_in = want_next && next_inside;
        uint32_t ns, ss;
        block_append2(app_out, want_shadow, &c->rays[cur][xcd].both, s_append, ns, ss);
        if (app_out) {
            ns = queue.slot(xcd, ns);
            nq_o[ns] = no;
            nq_d[ns] = nd;
        }
        uint32_t ni = block_append(app_in, &c->inside[cur][xcd].v, s_append);
        if (app_in) {
            ni = queue.slot(xcd, ni);
            niq_o[ni] = no;
            niq_d[ni] = nd;
        }
        if (want_shadow) {
            ss = queue.slot(xcd, ss);
            s_o[ss] = so;
            s_d[ss] = sd;
            s_c[ss] = sc;
        }
    }
    // object traces of this launch count as closest-hit rays
    for (int off = 32; off > 0; off >>= 1) inside_traces += __shfl_xor(inside_traces, off);
    if (__lane_id() == 0 && inside_traces) atomicAdd(&c->extension_rays, inside_traces);
}

static int ensure_wavefront(cupbr_renderer* r, uint32_t paths, uint32_t grid_threads) {
    Wavefront& wf = r->wf;
    int rc;
    if (paths > wf.capacity) {
        const size_t n = paths;
        if ((rc = wf.weight.ensure(n * 16))) return rc;
        if ((rc = wf.radiance.ensure(n * 16))) return rc;
        for (int k = 0; k < 2; ++k) {
            if ((rc = wf.q_o[k].ensure(n * 16))) return rc;
            if ((rc = wf.q_d[k].ensure(n * 16))) return rc;
        }
        if ((rc = wf.q_hit.ensure(n * 8))) return rc;
        for (int k = 0; k < 2; ++k) {
            if ((rc = wf.s_o[k].ensure(n * 16))) return rc;
            if ((rc = wf.s_d[k].ensure(n * 16))) return rc;
            if ((rc = wf.s_c[k].ensure(n * 16))) return rc;
        }
        wf.capacity = paths;
    }
    if ((rc = wf.counters.ensure(sizeof(Counters)))) return rc;
    const uint32_t entries = r->scene->stack_entries;
    if (entries > (uint32_t)kPtLds) {
        if ((rc = wf.spill.ensure((size_t)(entries - kPtLds) * grid_threads * 4))) return rc;
    }
    return CUPBR_OK;
}

// The queues' granules for batches of up to npath paths: 1024 rays, fewer where that would leave an XCD
// less than 8 of them (small images keep all XCDs busy)
static XcdQueue xcd_queue(uint32_t npath) {
    uint32_t lg = 10;
    while (lg > 6u && (npath >> lg) < 64u) --lg;
    return XcdQueue{lg};
}

// SampleOrder of a batch of nb frames of npix pixels: as many frames per wave as divide nb (a power
// of two up to 64) while 64 / frames still divides the pixel count
SampleOrder sample_order(uint32_t npix, uint32_t nb) {
    uint32_t f = 64;
    while (f > 1u && (nb % f != 0u || npix % (64u / f) != 0u)) f >>= 1;
    return SampleOrder{npix, nb, f};
}

int render_pathtracer(cupbr_renderer* r, const cupbr_camera& cam, uint32_t frame0, uint32_t spp) {
    const uint32_t w = r->width, h = r->height, npix = w * h;
    if (npix == 0 || spp == 0) return CUPBR_OK;
    const bool nrc = r->nrc != nullptr;
    // Paths in flight, in whole frames: up to 128M (200 B of path state and queues per path, so
    // up to ~27 GB). A trace launch ends with the last 64-ray chunks of its slowest waves, and
    // with more paths per launch that tail is a smaller share of it (1080p, 64 spp, Msamples/s:
    // 17 frames per batch 637, 32 frames 651, all 64 frames 656). Bounded to an eighth of the
    // device memory. A call of one frame (interactive use) holds one frame of paths. With a
    // radiance cache the same holds: a call of k frames is one batch, and the cache trains after
    // each batch.
    const uint32_t target = 1u << 27;
    uint32_t cap = 1u << 27;
    if (const size_t total = device_memory()) cap = (uint32_t)std::min<size_t>(cap, std::max<size_t>(total / 8 / 200, 1u << 20));
    uint32_t batch = std::max<uint32_t>(1, (target + npix - 1) / npix);
    batch = std::min(batch, std::max<uint32_t>(1, cap / npix));
    batch = std::min(batch, spp);
    const int blocks = device_cu_count() * 8;
    const uint32_t grid_threads = (uint32_t)blocks * kPtBlock;
    const XcdQueue queue = xcd_queue(batch * npix);
    int rc = ensure_wavefront(r, queue.capacity(batch * npix), grid_threads);
    if (rc) return rc;
    Wavefront& wf = r->wf;
    Counters* c = wf.counters.as<Counters>();
    CUPBR_HIP_CHECK(hipMemsetAsync(c, 0, sizeof(Counters), r->stream));
    r->counted = true;
    uint32_t* spill = r->scene->stack_entries > (uint32_t)kPtLds ? wf.spill.as<uint32_t>() : nullptr;
    const DevScene& S = r->scene->dev;
    float* img = r->images[CUPBR_IMAGE_OUTPUT].as<float>();
    const uint32_t bounces = std::max<uint32_t>(1, r->max_trace_depth);  // do { } while (depth < max)
    auto trace = r->counting ? k_pt_trace<true> : k_pt_trace<false>;
    // camera rays as wave packets (the visit-counting pass keeps the per-ray traversal, whose
    // counts define the algorithmic bytes of a trace launch)
    const bool packet = !r->counting && r->scene->stack_entries <= kPacketStack && S.n_nodes > 0;
    const bool pcg = r->rng == CUPBR_RNG_PCG;
    auto shade = nrc ? (pcg ? k_pt_shade_nrc<Pcg32> : k_pt_shade_nrc<uint32_t>)
                     : (pcg ? k_pt_shade<Pcg32> : k_pt_shade<uint32_t>);
    auto raygen = pcg ? k_pt_raygen<Pcg32> : k_pt_raygen<uint32_t>;
    auto camera = pcg ? k_pt_camera<Pcg32> : k_pt_camera<uint32_t>;
    const auto packet_blocks = [](uint32_t n) { return ((n + kPtBlock - 1) / kPtBlock + 7u) / 8u * 8u; };
    // a small batch in one launch (not when the stages of a frame are timed, and only as the call's one batch: the
    // kernel counts on from the call's cleared counters, where bounce 0 of the queues starts each batch at 0)
    const uint32_t cus = (uint32_t)device_cu_count();
    const bool deep = r->scene->stack_entries > kDeepStack;
    const bool whole = packet && !r->profiling && batch == spp &&
                       (size_t)batch * npix <= (size_t)cus * (deep || nrc ? kWholePaths : bounces > 1 ? kWholeShallow : kWholeShallowDirect);
    uint32_t per_wave = 8;
    while (per_wave < 64u && (size_t)per_wave * cus * (deep ? 16u : 8u) < (size_t)batch * npix) per_wave *= deep ? 2u : 8u;
    auto paths = nrc ? (pcg ? k_pt_paths<true, true, Pcg32> : k_pt_paths<true, true, uint32_t>)
                 : per_wave < 64u ? (pcg ? k_pt_paths<false, true, Pcg32> : k_pt_paths<false, true, uint32_t>)
                                  : (pcg ? k_pt_paths<false, false, Pcg32> : k_pt_paths<false, false, uint32_t>);
    NrcShade ns{nullptr, nullptr, 0, __builtin_inff()};
    uint32_t train_thresh = 0;
    const uint32_t path_blocks = packet_blocks((batch * npix + per_wave - 1) / per_wave * 64u);
    uint32_t part_rows = 0;  // whole paths: room for the rows of one XCD's paths, one a vertex
    if (nrc) {
        if (whole) part_rows = (uint32_t)std::min<size_t>(r->nrc_max_rows, (size_t)part_paths(path_blocks, per_wave) * bounces);
        if ((rc = r->nrc_queries.ensure((size_t)batch * npix * 80)) ||
            (rc = r->nrc_pending.ensure((size_t)(whole ? 8u * part_rows : r->nrc_max_rows) * 96)) ||
            (rc = r->nrc_rows.ensure((size_t)r->nrc_max_rows * 80)))
            return rc;
        ns = NrcShade{r->nrc_queries.as<float4>(), r->nrc_pending.as<float4>(), whole ? part_rows : r->nrc_max_rows,
                      r->nrc_camera_min_roughness};
        if (!r->side_stream) {
            if (hipStreamCreateWithFlags(&r->side_stream, hipStreamNonBlocking) != hipSuccess ||
                hipEventCreateWithFlags(&r->ev_queries, hipEventDisableTiming) != hipSuccess ||
                hipEventCreateWithFlags(&r->ev_side_done, hipEventDisableTiming) != hipSuccess)
                return set_error(CUPBR_ERR_HIP, "could not create the radiance cache's stream");
        }
        const double frac = std::min(1.0, (double)r->nrc_train_paths / (double)npix);
        train_thresh = frac >= 1.0 ? 0xFFFFFFFFu : (uint32_t)(frac * 4294967296.0);
    }
    if ((rc = stage_mark(r, -1))) return rc;
    for (uint32_t s0 = 0; s0 < spp; s0 += batch) {
        const uint32_t nb = std::min(batch, spp - s0);
        bool side_pending = false;  // cache inference of this batch running on the side stream
        const uint32_t npath = nb * npix;
        const SampleOrder order = sample_order(npix, nb);
        // with camera packets, bounce 0 makes its own camera rays (k_pt_camera)
        if (!packet) {
            hipLaunchKernelGGL(raygen, dim3((npath + kPtBlock - 1) / kPtBlock), dim3(kPtBlock), 0, r->stream, cam, w,
                               h, frame0 + s0, npath, order, wf.q_o[0].as<float4>(), wf.q_d[0].as<float4>(),
                               wf.weight.as<float4>(), wf.radiance.as<float4>(), c, queue, train_thresh);
            if ((rc = stage_mark(r, 3))) return rc;
        }
        if (whole)
            hipLaunchKernelGGL(paths, dim3(path_blocks), dim3(kPtBlock), 0,
                               r->stream, S, npath, per_wave, cam, w, h,
                               frame0 + s0, order, train_thresh, r->max_trace_depth, (int)r->russian_roulette,
                               wf.radiance.as<float4>(), c, ns, spill, grid_threads);
        // per bounce: trace (this bounce's extension rays + the previous bounce's shadow rays), then
        // shade (appends the next extension rays and this bounce's shadow rays, by bounce parity)
        for (uint32_t b = 0; b <= bounces && !whole; ++b) {
            const int cur = (int)(b & 1);
            if (b == 0 && packet) {
                hipLaunchKernelGGL(camera, dim3(packet_blocks(npath)), dim3(kPtBlock), 0, r->stream, S, npath, cam, w,
                                   h, frame0 + s0, order, train_thresh, wf.q_o[0].as<float4>(), wf.q_d[0].as<float4>(), wf.radiance.as<float4>(), wf.q_hit.as<float2>(), c, queue);
            } else {
                hipLaunchKernelGGL(trace, dim3(blocks), dim3(kPtBlock), 0, r->stream, S, cur, wf.q_o[cur].as<float4>(),
                                   wf.q_d[cur].as<float4>(), wf.q_hit.as<float2>(), wf.s_o[cur ^ 1].as<float4>(),
                                   wf.s_d[cur ^ 1].as<float4>(), wf.s_c[cur ^ 1].as<float4>(),
                                   wf.radiance.as<float4>(), c, queue, spill, grid_threads);
            }
            if ((rc = stage_mark(r, 0))) return rc;
            if (b == bounces) break;  // the last trace only had the last bounce's shadow rays
            hipLaunchKernelGGL(shade, dim3(blocks), dim3(kPtBlock), 0, r->stream, S, cur, b, r->max_trace_depth,
                               (int)r->russian_roulette, wf.q_o[cur].as<float4>(),
                               wf.q_d[cur].as<float4>(), wf.q_hit.as<float2>(), wf.q_o[cur ^ 1].as<float4>(),
                               wf.q_d[cur ^ 1].as<float4>(), wf.s_o[cur].as<float4>(), wf.s_d[cur].as<float4>(),
                               wf.s_c[cur].as<float4>(), wf.weight.as<float4>(), wf.radiance.as<float4>(), c, queue,
                               ns, b == 0 && packet ? 0u : ~0u);
            if ((rc = stage_mark(r, 1))) return rc;
            if (nrc && b == 1 && bounces > 2 && npath >= kSidePaths) {
                // The paths that queried the cache so far have no shadow ray left in flight (the
                // shadow rays of bounce 0 were traced before this shade, and a query vertex
                // traces none), and no later kernel touches their radiance until the final pass
                // below: their inference runs on the side stream while the remaining bounces
                // (mostly training paths) are traced.
                hipLaunchKernelGGL(k_snapshot_queries, dim3(1), dim3(1), 0, r->stream, c);
                CUPBR_HIP_CHECK(hipEventRecord(r->ev_queries, r->stream));
                CUPBR_HIP_CHECK(hipStreamWaitEvent(r->side_stream, r->ev_queries, 0));
                if ((rc = nrc_infer(r->nrc, r->nrc_queries.as<float>(), npath,
                                    &c->query_early.v, 20,
                                    wf.radiance.as<float>(), true, r->side_stream)))
                    return rc;
                CUPBR_HIP_CHECK(hipEventRecord(r->ev_side_done, r->side_stream));
                side_pending = true;
            }
        }
        if (nrc) {
            // throughput * cache for the paths that ended at a cache vertex (those not already
            // inferred on the side stream), then the training rows
            const uint32_t* n_queries = whole ? &c->cache_part[0].queries : &c->cache.queries;
            const NrcParts parts = whole ? NrcParts{part_paths(path_blocks, per_wave), (uint32_t)(sizeof c->cache_part[0] / 4)} : NrcParts{};
            if ((rc = nrc_infer(r->nrc, r->nrc_queries.as<float>(), npath, n_queries, 20, wf.radiance.as<float>(), true,
                                r->stream, side_pending ? &c->query_early.v : nullptr, parts)))
                return rc;
            if (side_pending) {
                CUPBR_HIP_CHECK(hipStreamWaitEvent(r->stream, r->ev_side_done, 0));
                side_pending = false;
            }
            if ((rc = stage_mark(r, 3))) return rc;
            const uint32_t pix_blocks = (npix + kPtBlock - 1) / kPtBlock;
            hipLaunchKernelGGL(k_accumulate_rows, dim3(pix_blocks + (uint32_t)device_cu_count()), dim3(kPtBlock), 0,
                               r->stream, img, wf.radiance.as<float4>(), w, h, order, frame0 + s0, nb, pix_blocks,
                               r->nrc_pending.as<float4>(), c, r->nrc_max_rows, part_rows, r->nrc_rows.as<float4>());
        } else {
            hipLaunchKernelGGL(k_accumulate, dim3((npix + kPtBlock - 1) / kPtBlock), dim3(kPtBlock), 0, r->stream, img,
                               wf.radiance.as<float4>(), w, h, order, frame0 + s0, nb);
        }
        if ((rc = stage_mark(r, 3))) return rc;
        // the row count stays on the device: a batch without training rows takes no steps (Cornell box,
        // 256x256, 1 spp and 4 steps: 0.83 -> 0.80 ms without the copy to the host and the wait for it)
        if (nrc && train_thresh != 0u && r->nrc_steps > 0) {
            if ((rc = nrc_train(r->nrc, r->nrc_rows.as<float>(), r->nrc_max_rows, r->nrc_batch, r->nrc_steps, r->nrc_lr,
                                nullptr, r->stream, &c->cache.rows)))
                return rc;
        }
        if (nrc && (rc = stage_mark(r, 3))) return rc;
    }
    CUPBR_HIP_CHECK(hipGetLastError());
    return CUPBR_OK;
}

int volume_paths_wavefront(cupbr_renderer* r, const cupbr_camera& cam, uint32_t frame0, uint32_t spp) {
    const uint32_t w = r->width, h = r->height, npix = w * h;
    if (npix == 0 || spp == 0) return CUPBR_OK;
    const uint32_t target = 1u << 27;
    uint32_t cap = 1u << 27;
    if (const size_t total = device_memory()) cap = (uint32_t)std::min<size_t>(cap, std::max<size_t>(total / 8 / 264, 1u << 20));
    uint32_t batch = std::max<uint32_t>(1, (target + npix - 1) / npix);
    batch = std::min(batch, std::max<uint32_t>(1, cap / npix));
    batch = std::min(batch, spp);
    const int blocks = device_cu_count() * 8;
    const uint32_t grid_threads = (uint32_t)blocks * kPtBlock;
    const XcdQueue queue = xcd_queue(batch * npix);
    int rc = ensure_wavefront(r, queue.capacity(batch * npix), grid_threads);
    if (rc) return rc;
    Wavefront& wf = r->wf;
    const uint32_t slots = queue.capacity(batch * npix);
    if (wf.iq_capacity < slots) {
        for (int k = 0; k < 2; ++k) {
            if ((rc = wf.iq_o[k].ensure((size_t)slots * 16)) || (rc = wf.iq_d[k].ensure((size_t)slots * 16))) return rc;
        }
        wf.iq_capacity = slots;
    }
    Counters* c = wf.counters.as<Counters>();
    CUPBR_HIP_CHECK(hipMemsetAsync(c, 0, sizeof(Counters), r->stream));
    r->counted = true;
    uint32_t* spill = r->scene->stack_entries > (uint32_t)kPtLds ? wf.spill.as<uint32_t>() : nullptr;
    const DevScene& S = r->scene->dev;
    float* img = r->images[CUPBR_IMAGE_OUTPUT].as<float>();
    const uint32_t bounces = std::max<uint32_t>(1, r->max_trace_depth);
    auto trace = r->counting ? k_pt_trace<true> : k_pt_trace<false>;
    const bool packet = !r->counting && r->scene->stack_entries <= kPacketStack && S.n_nodes > 0;
    if ((rc = stage_mark(r, -1))) return rc;
    for (uint32_t s0 = 0; s0 < spp; s0 += batch) {
        const uint32_t nb = std::min(batch, spp - s0);
        const uint32_t npath = nb * npix;
        // the path tracer's ray generation (camera rays in SampleOrder), seed tea<4>(pixel, frame)
        // (VolumeRenderer.cu:229-234); rad[p].w = 0: outside every object
        // (VolumeRenderer.cu:229-234), made inside the camera trace with camera packets
        const SampleOrder order = sample_order(npix, nb);
        if (!packet) {
            hipLaunchKernelGGL(k_pt_raygen<uint32_t>, dim3((npath + kPtBlock - 1) / kPtBlock), dim3(kPtBlock), 0,
                               r->stream, cam, w, h, frame0 + s0, npath, order, wf.q_o[0].as<float4>(),
                               wf.q_d[0].as<float4>(), wf.weight.as<float4>(), wf.radiance.as<float4>(), c, queue, 0u);
            if ((rc = stage_mark(r, 3))) return rc;
        }
        for (uint32_t b = 0; b <= bounces; ++b) {
            const int cur = (int)(b & 1);
            if (b == 0 && packet) {
                const uint32_t nblk = (npath + kPtBlock - 1) / kPtBlock;
                hipLaunchKernelGGL(k_pt_camera<uint32_t>, dim3((nblk + 7u) / 8u * 8u), dim3(kPtBlock), 0, r->stream, S,
                                   npath, cam, w, h, frame0 + s0, order, 0u, wf.q_o[0].as<float4>(),
                                   wf.q_d[0].as<float4>(), wf.radiance.as<float4>(),
                                   wf.q_hit.as<float2>(), c, queue);
            } else {
                hipLaunchKernelGGL(trace, dim3(blocks), dim3(kPtBlock), 0, r->stream, S, cur, wf.q_o[cur].as<float4>(),
                                   wf.q_d[cur].as<float4>(), wf.q_hit.as<float2>(), wf.s_o[cur ^ 1].as<float4>(),
                                   wf.s_d[cur ^ 1].as<float4>(), wf.s_c[cur ^ 1].as<float4>(),
                                   wf.radiance.as<float4>(), c, queue, spill, grid_threads);
            }
            if ((rc = stage_mark(r, 0))) return rc;
            if (b == bounces) break;
            hipLaunchKernelGGL(k_vol_shade, dim3(blocks), dim3(kPtBlock), 0, r->stream, S, cur, b, r->max_trace_depth,
                               (int)r->russian_roulette, wf.q_o[cur].as<float4>(),
                               wf.q_d[cur].as<float4>(),
                               wf.q_hit.as<float2>(), wf.iq_o[cur].as<float4>(), wf.iq_d[cur].as<float4>(),
                               wf.q_o[cur ^ 1].as<float4>(), wf.q_d[cur ^ 1].as<float4>(),
                               wf.iq_o[cur ^ 1].as<float4>(), wf.iq_d[cur ^ 1].as<float4>(), wf.s_o[cur].as<float4>(),
                               wf.s_d[cur].as<float4>(), wf.s_c[cur].as<float4>(), wf.weight.as<float4>(),
                               wf.radiance.as<float4>(), c, queue, b == 0 && packet ? 0u : ~0u);
            if ((rc = stage_mark(r, 1))) return rc;
        }
        hipLaunchKernelGGL(k_accumulate, dim3((npix + kPtBlock - 1) / kPtBlock), dim3(kPtBlock), 0, r->stream, img,
                           wf.radiance.as<float4>(), w, h, order, frame0 + s0, nb);
        if ((rc = stage_mark(r, 3))) return rc;
    }
    CUPBR_HIP_CHECK(hipGetLastError());
    return CUPBR_OK;
}

int gdpt_paths_wavefront(cupbr_renderer* r, const cupbr_camera& cam, uint32_t frame0, uint32_t spp) {
    const uint32_t w = r->width, h = r->height;
    if (w < 3 || h < 3 || spp == 0) return CUPBR_OK;  // no interior pixel: the buffers stay as they are
    const uint32_t n_int = (w - 2u) * (h - 2u);
    // paths in flight, in whole frames (5 per interior pixel), bounded as in the path tracer
    const uint32_t target = 1u << 27;
    uint32_t cap = 1u << 27;
    if (const size_t total = device_memory()) cap = (uint32_t)std::min<size_t>(cap, std::max<size_t>(total / 8 / 200, 1u << 20));
    const uint32_t per_frame = 5u * n_int;
    uint32_t batch = std::max<uint32_t>(1, target / per_frame);
    batch = std::min(batch, std::max<uint32_t>(1, cap / per_frame));
    batch = std::min(batch, spp);
    const int blocks = device_cu_count() * 8;
    const uint32_t grid_threads = (uint32_t)blocks * kPtBlock;
    const XcdQueue queue = xcd_queue(batch * per_frame);
    int rc = ensure_wavefront(r, queue.capacity(batch * per_frame), grid_threads);
    if (rc) return rc;
    Wavefront& wf = r->wf;
    if ((rc = wf.gdpt_slot.ensure((size_t)2 * batch * n_int * sizeof(uint32_t)))) return rc;
    uint32_t* slots[2] = {wf.gdpt_slot.as<uint32_t>(), wf.gdpt_slot.as<uint32_t>() + (size_t)batch * n_int};
    Counters* c = wf.counters.as<Counters>();
    CUPBR_HIP_CHECK(hipMemsetAsync(c, 0, sizeof(Counters), r->stream));
    r->counted = true;
    uint32_t* spill = r->scene->stack_entries > (uint32_t)kPtLds ? wf.spill.as<uint32_t>() : nullptr;
    const DevScene& S = r->scene->dev;
    float* im[kNumImages];
    for (int k = 0; k < kNumImages; ++k) im[k] = r->images[k].as<float>();
    const uint32_t bounces = std::max<uint32_t>(1, r->max_trace_depth);
    auto trace = r->counting ? k_pt_trace<true> : k_pt_trace<false>;
    const bool packet = !r->counting && r->scene->stack_entries <= kPacketStack && S.n_nodes > 0;
    if ((rc = stage_mark(r, -1))) return rc;
    for (uint32_t s0 = 0; s0 < spp; s0 += batch) {
        const uint32_t nb = std::min(batch, spp - s0);
        const uint32_t groups = nb * n_int, npath = 5u * groups;
        if (!packet) {  // with camera packets the camera trace makes the rays (k_gdpt_camera)
            hipLaunchKernelGGL(k_gdpt_raygen, dim3((npath + kPtBlock - 1) / kPtBlock), dim3(kPtBlock), 0, r->stream,
                               cam, w, h, frame0 + s0, n_int, groups, wf.q_o[0].as<float4>(), wf.q_d[0].as<float4>(),
                               wf.weight.as<float4>(), wf.radiance.as<float4>(), slots[0], c, queue);
            if ((rc = stage_mark(r, 3))) return rc;
        }
        for (uint32_t b = 0; b <= bounces; ++b) {
            const int cur = (int)(b & 1);
            if (b == 0 && packet) {
                const uint32_t nblk = (npath + kPtBlock - 1) / kPtBlock;
                hipLaunchKernelGGL(k_gdpt_camera, dim3((nblk + 7u) / 8u * 8u), dim3(kPtBlock), 0, r->stream, S, npath,
                                   cam, w, h, frame0 + s0, n_int, wf.q_o[0].as<float4>(), wf.q_d[0].as<float4>(),
                                   wf.radiance.as<float4>(), slots[0], wf.q_hit.as<float2>(), c, queue);
            } else {
                hipLaunchKernelGGL(trace, dim3(blocks), dim3(kPtBlock), 0, r->stream, S, cur, wf.q_o[cur].as<float4>(),
                                   wf.q_d[cur].as<float4>(), wf.q_hit.as<float2>(), wf.s_o[cur ^ 1].as<float4>(),
                                   wf.s_d[cur ^ 1].as<float4>(), wf.s_c[cur ^ 1].as<float4>(),
                                   wf.radiance.as<float4>(), c, queue, spill, grid_threads);
            }
            if ((rc = stage_mark(r, 0))) return rc;
            if (b == bounces) break;
            hipLaunchKernelGGL(k_gdpt_shade, dim3(blocks), dim3(kPtBlock), 0, r->stream, S, cur, b, r->max_trace_depth,
                               wf.q_o[cur].as<float4>(), wf.q_d[cur].as<float4>(),
                               wf.q_hit.as<float2>(), wf.q_o[cur ^ 1].as<float4>(), wf.q_d[cur ^ 1].as<float4>(),
                               wf.s_o[cur].as<float4>(), wf.s_d[cur].as<float4>(), wf.s_c[cur].as<float4>(),
                               wf.weight.as<float4>(), wf.radiance.as<float4>(), c, queue, slots[b & 1],
                               slots[(b + 1) & 1], b == 0 && packet ? 0u : ~0u);
            if ((rc = stage_mark(r, 1))) return rc;
        }
        hipLaunchKernelGGL(k_gdpt_accumulate, dim3((n_int + kPtBlock - 1) / kPtBlock), dim3(kPtBlock), 0, r->stream,
                           im[CUPBR_IMAGE_BASE], im[CUPBR_IMAGE_GRADIENT_X_FORWARD], im[CUPBR_IMAGE_GRADIENT_X_BACKWARD],
                           im[CUPBR_IMAGE_GRADIENT_Y_FORWARD], im[CUPBR_IMAGE_GRADIENT_Y_BACKWARD],
                           wf.radiance.as<float4>(), w, h, n_int, frame0 + s0, nb);
        if ((rc = stage_mark(r, 3))) return rc;
    }
    CUPBR_HIP_CHECK(hipGetLastError());
    return CUPBR_OK;
}

}  // namespace cupbr
