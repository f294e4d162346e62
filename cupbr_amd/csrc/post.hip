// Bloom and tone mapping.
//
// The reference builds a 6-level pyramid in 13 launches (PostProcessor.cpp:125-142,
// PyramidConstructor.cu:9-169), but its upsampling reads the *down* pyramid
// (`up[i] = tent(down[i+1])/16 + down[i]`, :79-80,111), so the output depends on
// levels 0 and 1 only:
//     out(p) = hdr(p) + ( tent3x3(down1)(p/2) / 16 + down0(p) )
//     down0  = threshold(hdr),  down1(q) = box2x2(down0)(2q)   (edge-clamped)
// This file computes exactly that, in the reference's FP32 operation order, in
// one pass per 64x8 tile: the tile's 34x6 block of down1 (with its one-texel
// halo) is built in LDS from hdr reads, then every output pixel reads its own
// hdr value again (an L1/L2 hit). A tile's reads reach 2 pixels into each
// neighbouring tile, so tiles are assigned to XCDs in contiguous row-major
// bands: the neighbours run on the same XCD at about the same time and their
// shared lines come from that XCD's L2. HBM traffic is then about one FP32 RGB
// read and one write per pixel (+ 4 bytes when the RGBA8 tone map is fused in).
#include <cstdio>
#include <vector>

#include "post.h"
#include "vecmath.h"

namespace cupbr {

constexpr int kTileW = 64, kTileH = 8;
constexpr int kD1W = kTileW / 2 + 2, kD1H = kTileH / 2 + 2;

// thresholding_kernel, PyramidConstructor.cu:9-30
__device__ __forceinline__ v3 threshold_px(v3 c, float4 t) {
    float b = c.x > c.y ? c.x : c.y;
    b = c.z > b ? c.z : b;
    float rq = clampf(b - t.y, 0.0f, t.z);
    rq = t.w * rq * rq;
    const float s = fmaxf(rq, b - t.x) / fmaxf(b, 1e-5f);
    return v3{c.x * s, c.y * s, c.z * s};
}

__device__ __forceinline__ uint8_t to_byte(float m) { return (uint8_t)(clampf(m, 0.0f, 1.0f) * 255.0f); }

// One channel of a power curve, to_byte(scale * powf(x, g) + shift). powf's 100 and more instructions, three times
// a pixel, bounded the tone map, so the byte is decided by the hardware's log2 and exp2 unless y lies within 2^-13 of
// a step, where powf is called. The error of y before its last roundings is below 255 * 1.055 (ln 2 * 0.53 * 2^-22 +
// 2^-23) = 6e-5 (relative errors of 2^-23 of either function and 2^-24 of the product, 0.53 being the largest
// |t| 2^t for t <= 0); the roundings of scale, shift and the factor 255 on both sides and powf's own last place are of
// the same size together, so that the 1.2e-4 of the margin is no proof: that the bytes are powf's for every float
// is checked by going through them all (k_tone_byte_check). The fused combine and tone map of 1080p: 39 -> 24 us.
__device__ __forceinline__ uint8_t power_byte(float x, float g, float scale, float shift) {
    constexpr float kStep = 1.0f / 8192.0f;
    if (x == 0.0f || x == 1.0f) return to_byte(scale * x + shift);  // black, saturated
    const float y = 255.0f * (scale * __builtin_amdgcn_exp2f(g * __builtin_amdgcn_logf(x)) + shift);
    if (x >= 1.0f && y >= 255.0f + kStep) return 255;
    const float k = floorf(y);
    if (x >= 1e-30f && x < 1.0f && y - k >= kStep && k + 1.0f - y >= kStep && y > 0.0f && y < 255.0f) return (uint8_t)k;
    return to_byte(scale * powf(x, g) + shift);
}

// reinhard_kernel / gamma_kernel, ToneMapper.cu:17-69 (truncating casts; 1.0 - expf() and the
// blue channel's 1.0f/2.2 are double expressions in the reference)
__device__ __forceinline__ uchar4 tonemap_px(v3 c, int32_t type, float exposure) {
    uint8_t m[3];
    const float cc[3] = {c.x, c.y, c.z};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        if (type == CUPBR_REINHARD) {
            // 1.0f - e is the double difference rounded to float: exact in double from e = 2^-29 on, 1 below
            const float base = 1.0f - expf(-cc[k] * exposure);
            m[k] = power_byte(base, k == 2 ? (float)(1.0f / 2.2) : 1.0f / 2.2f, 1.0f, 0.0f);
        } else if (type == CUPBR_ACES) {  // Narkowicz's ACES filmic fit, then gamma 1/2.2
            const float x = cc[k] * exposure;
            const float f = (x * (2.51f * x + 0.03f)) / (x * (2.43f * x + 0.59f) + 0.14f);
            m[k] = power_byte(clampf(f, 0.0f, 1.0f), 1.0f / 2.2f, 1.0f, 0.0f);
        } else {
            const float x = cc[k];
            m[k] = x <= 0.0031308f ? to_byte(12.92f * x) : power_byte(x, 1.0f / 2.4f, 1.055f, -0.055f);
        }
    }
    return make_uchar4(m[0], m[1], m[2], 255);
}

__device__ __forceinline__ v3 ld_px(const float* img, uint32_t w, int x, int y) {
    return ld3(img + 3 * ((size_t)y * w + x));
}

__global__ __launch_bounds__(256) void k_bloom(const float* __restrict__ hdr, float* __restrict__ out,
                                               uchar4* __restrict__ rgba, uint32_t w, uint32_t h, float4 curve,
                                               int32_t type, float exposure) {
    __shared__ float d1[3][kD1H][kD1W];
    // workgroups are dispatched to the 8 XCDs round-robin by block id: block b runs on XCD b % 8,
    // which takes tiles [xcd * q + min(xcd, r), ... + its block count) in row-major order
    // (a bijection onto the n tiles: XCD x has q + (x < r) blocks)
    const uint32_t n = gridDim.x, q = n / 8u, rem = n % 8u, xcd = blockIdx.x % 8u;
    const uint32_t tile = xcd * q + (xcd < rem ? xcd : rem) + blockIdx.x / 8u;
    const uint32_t tiles_x = (w + kTileW - 1) / kTileW;
    const int x0 = (int)(tile % tiles_x) * kTileW, y0 = (int)(tile / tiles_x) * kTileH;
    const int w1 = (int)(w / 2), h1 = (int)(h / 2);
    const int qx0 = x0 / 2 - 1, qy0 = y0 / 2 - 1;
    const int tid = threadIdx.x;
    if (tid < kD1W * kD1H) {
        const int j = tid / kD1W, i = tid - j * kD1W;
        int qx = qx0 + i, qy = qy0 + j;
        qx = qx < 0 ? 0 : (qx >= w1 ? w1 - 1 : qx);  // upscale_and_combine_kernel :101-104
        qy = qy < 0 ? 0 : (qy >= h1 ? h1 - 1 : qy);
        v3 r = splat(0.0f);
#pragma unroll
        for (int k = 0; k < 4; ++k) {  // downsample_kernel :51-64, reads (0,0),(0,1),(1,0),(1,1)
            int sx = 2 * qx + (k >> 1), sy = 2 * qy + (k & 1);
            if (sx >= (int)w) sx = (int)w - 1;
            if (sy >= (int)h) sy = (int)h - 1;
            r += threshold_px(ld_px(hdr, w, sx, sy), curve);
        }
        r = r / 4.0f;
        d1[0][j][i] = r.x;
        d1[1][j][i] = r.y;
        d1[2][j][i] = r.z;
    }
    __syncthreads();
    const int tx = tid & (kTileW - 1);
#pragma unroll
    for (int row = 0; row < kTileH; row += 256 / kTileW) {
        const int x = x0 + tx, y = y0 + row + tid / kTileW;
        if (x >= (int)w || y >= (int)h) continue;
        const v3 c = ld_px(hdr, w, x, y);
        const v3 d0 = threshold_px(c, curve);
        const int cx = x / 2 - qx0, cy = y / 2 - qy0;
        v3 res = splat(0.0f);
        const float kw[3] = {1.0f, 2.0f, 1.0f};
#pragma unroll
        for (int u = -1; u < 2; ++u)
#pragma unroll
            for (int v = -1; v < 2; ++v) {
                const float k = kw[u + 1] * kw[v + 1];
                res += v3{d1[0][cy + v][cx + u], d1[1][cy + v][cx + u], d1[2][cy + v][cx + u]} * k;
            }
        const v3 up0 = res / 16.0f + d0;  // :111
        const v3 o = c + up0;             // combine_kernel :124
        st3(out + 3 * ((size_t)y * w + x), o);
        if (rgba) rgba[(size_t)y * w + x] = tonemap_px(o, type, exposure);
    }
}

__global__ __launch_bounds__(256) void k_tonemap(const float* __restrict__ hdr, uchar4* __restrict__ rgba, size_t n,
                                                 int32_t type, float exposure) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    rgba[i] = tonemap_px(ld3(hdr + 3 * i), type, exposure);
}

// ------------------------------------------------------------------ Gaussian pyramid bloom
// (CUPBR_BLOOM_GAUSSIAN5, an addition: see cupbr_post_set_bloom_pyramid for the definition.) What bounds it is
// one read and one write of the image, and below that the launches: a level of a 1080p image is a few
// microseconds of latency whatever its size. So four launches: level 1 from the image (the threshold is
// recomputed where it is read), levels 2 and 3, levels 4 and 5 (a block computes the part of the middle level
// that its tile needs), and the image, whose blocks walk up the pyramid from level 5 for their own tile in
// LDS. A 1080p frame with the tone map: 85 us with one launch
// per level and pass (11), 53 with these (11, 6, 4 and 24 us of kernels; the copy rate allows 12).

struct LevelDims {
    uint32_t w, h;
};

// One blur and 2:1 decimation in LDS: dst(x, y) = blur(src)(2x, 2y), rows of five taps [1 4 6 4 1] summed
// first, then the five rows, then / 256. src: sh rows of kSrc texels; the blur of column i starts at texel
// col(i), that of row j at row(j); rows: scratch of sh x dw texels.
__device__ __forceinline__ v3 lds_px(const float* p) { return mk(p[0], p[1], p[2]); }
__device__ __forceinline__ void lds_put(float* p, v3 v) {
    p[0] = v.x;
    p[1] = v.y;
    p[2] = v.z;
}
template <int kSrcW, int kSrcH, int kDstW, int kDstH, class Col, class Row, class Put>
__device__ __forceinline__ void gauss_down(const float* src, float* rows, Col col, Row row, Put put) {
    const float wt[5] = {1.0f, 4.0f, 6.0f, 4.0f, 1.0f};
    for (int k = threadIdx.x; k < kSrcH * kDstW; k += 256) {
        const int j = k / kDstW, i = k - j * kDstW;
        const float* p = src + 3 * (j * kSrcW + col(i));
        v3 r = splat(0.0f);
#pragma unroll
        for (int t = 0; t < 5; ++t) r += lds_px(p + 3 * t) * wt[t];
        lds_put(rows + 3 * k, r);
    }
    __syncthreads();
    for (int k = threadIdx.x; k < kDstH * kDstW; k += 256) {
        const int j = k / kDstW, i = k - j * kDstW;
        const float* p = rows + 3 * (row(j) * kDstW + i);
        v3 acc = splat(0.0f);
#pragma unroll
        for (int t = 0; t < 5; ++t) acc += lds_px(p + 3 * t * kDstW) * wt[t];
        put(i, j, acc / 256.0f);
    }
}

// texels [x0, x0 + kW) x [y0, y0 + kH) of an image, edge-clamped: a thread's share, all loads in flight at once,
// and their place in LDS
template <int kW, int kH>
struct Tile {
    static constexpr int kEach = (kW * kH + 255) / 256;
    v3 v[kEach];
    __device__ __forceinline__ void load(const float* __restrict__ img, LevelDims d, int x0, int y0) {
#pragma unroll
        for (int e = 0; e < kEach; ++e) {
            const int k = min((int)threadIdx.x + e * 256, kW * kH - 1), j = k / kW, i = k - j * kW;
            v[e] = ld_px(img, d.w, min(max(x0 + i, 0), (int)d.w - 1), min(max(y0 + j, 0), (int)d.h - 1));
        }
    }
    template <class Map>
    __device__ __forceinline__ void store(float* lds, Map map) const {
#pragma unroll
        for (int e = 0; e < kEach; ++e) {
            const int k = threadIdx.x + e * 256;
            if (k < kW * kH) lds_put(lds + 3 * k, map(v[e]));
        }
    }
    __device__ __forceinline__ void store(float* lds) const {
        store(lds, [](v3 c) { return c; });
    }
};

// level 1: tiles of 32 x 8 texels from 67 x 19 pixels
__global__ __launch_bounds__(256) void k_gauss_first(const float* __restrict__ hdr, LevelDims d0, float* __restrict__ l1,
                                                     LevelDims d1, float4 curve) {
    __shared__ float src[67 * 19 * 3], rows[32 * 19 * 3];
    const int x0 = blockIdx.x * 32, y0 = blockIdx.y * 8;
    Tile<67, 19> tile;
    tile.load(hdr, d0, 2 * x0 - 2, 2 * y0 - 2);
    tile.store(src, [&](v3 c) { return threshold_px(c, curve); });
    __syncthreads();
    gauss_down<67, 19, 32, 8>(
        src, rows, [](int i) { return 2 * i; }, [](int j) { return 2 * j; },
        [&](int i, int j, v3 v) {
            const uint32_t x = x0 + i, y = y0 + j;
            if (x < d1.w && y < d1.h) st3(l1 + 3 * ((size_t)y * d1.w + x), v);
        });
}

// Two levels: tiles of kT x kT texels of the lower one (dst) from the 2 kT + 3 texels a side of the level between
// (mid) that they blur, and those from 4 kT + 9 of src; a block writes the 2 kT x 2 kT of mid above its tile.
template <int kT>
__global__ __launch_bounds__(256) void k_gauss_two(const float* __restrict__ src, LevelDims ds, float* __restrict__ mid,
                                                   LevelDims dm, float* __restrict__ dst, LevelDims dd) {
    constexpr int kM = 2 * kT + 3, kS = 2 * kM + 3;
    __shared__ float s[kS * kS * 3], rows[kS * kM * 3], m[kM * kM * 3], mrows[kM * kT * 3];
    const int x0 = blockIdx.x * kT, y0 = blockIdx.y * kT;
    const int mx0 = 2 * x0 - 2, my0 = 2 * y0 - 2, sx0 = 2 * mx0 - 2, sy0 = 2 * my0 - 2;
    Tile<kS, kS> tile;
    tile.load(src, ds, sx0, sy0);
    tile.store(s);
    __syncthreads();
    const auto mx = [&](int i) { return min(max(mx0 + i, 0), (int)dm.w - 1); };  // mid's edge-clamped coordinates
    const auto my = [&](int j) { return min(max(my0 + j, 0), (int)dm.h - 1); };
    gauss_down<kS, kS, kM, kM>(
        s, rows, [&](int i) { return 2 * mx(i) - 2 - sx0; }, [&](int j) { return 2 * my(j) - 2 - sy0; },
        [&](int i, int j, v3 v) {
            lds_put(m + 3 * (j * kM + i), v);
            const int x = mx0 + i, y = my0 + j;
            if (i >= 2 && i < 2 + 2 * kT && j >= 2 && j < 2 + 2 * kT && x < (int)dm.w && y < (int)dm.h)
                st3(mid + 3 * ((size_t)y * dm.w + x), v);
        });
    __syncthreads();
    gauss_down<kM, kM, kT, kT>(
        m, mrows, [](int i) { return 2 * i; }, [](int j) { return 2 * j; },
        [&](int i, int j, v3 v) {
            const uint32_t x = x0 + i, y = y0 + j;
            if (x < dd.w && y < dd.h) st3(dst + 3 * ((size_t)y * dd.w + x), v);
        });
}

// A coarse level (the texels from (cx0, cy0) in LDS, kW a row; d its size) sampled at fine texel (x, y): the texel
// (x/2, y/2), the mean of two texels along an odd coordinate (edge-clamped)
template <int kW>
__device__ __forceinline__ v3 gauss_up(const float* coarse, uint32_t cx0, uint32_t cy0, LevelDims d, uint32_t x, uint32_t y) {
    const uint32_t x0 = x >> 1, y0 = y >> 1;
    const uint32_t x1 = (x & 1u) ? min(x0 + 1u, d.w - 1u) : x0, y1 = (y & 1u) ? min(y0 + 1u, d.h - 1u) : y0;
    const auto at = [&](uint32_t cx, uint32_t cy) { return lds_px(coarse + 3 * ((cy - cy0) * kW + (cx - cx0))); };
    return ((at(x0, y0) + at(x1, y0)) * 0.5f + (at(x0, y1) + at(x1, y1)) * 0.5f) * 0.5f;
}

// U_k = L_k + up(U_{k+1}), in place, for the kW x kH texels of level k in LDS
template <int kW, int kH, int kCoarseW>
__device__ __forceinline__ void gauss_up_tile(float* fine, uint32_t x0, uint32_t y0, LevelDims df, const float* coarse,
                                              uint32_t cx0, uint32_t cy0, LevelDims dc) {
    for (int k = threadIdx.x; k < kW * kH; k += 256) {
        const int j = k / kW, i = k - j * kW;
        const uint32_t x = min(x0 + i, df.w - 1u), y = min(y0 + j, df.h - 1u);
        lds_put(fine + 3 * k, lds_px(fine + 3 * k) + gauss_up<kCoarseW>(coarse, cx0, cy0, dc, x, y));
    }
    __syncthreads();
}

struct Pyramid {
    const float* level[kGaussLevels + 1];
    LevelDims dim[kGaussLevels + 1];
};

constexpr uint32_t kCombineRows = 4;  // of a thread's column (8: half the blocks, 59 against 53 us a frame)

// out = hdr + (L0 + up(U1)) / 6, with the tone map fused when rgba is given: tiles of 64 x 4 kCombineRows pixels. The
// rows needed of the coarser levels: half of the finer one's and one more, from half of its first row on; a first
// row is even (a multiple of 16 >> level) except in the last levels, where half rounded down and one more is two
// rows for an even first row and for an odd one.
__global__ __launch_bounds__(256) void k_gauss_combine(const float* __restrict__ hdr, Pyramid P, float4 curve,
                                                       float* __restrict__ out, uchar4* __restrict__ rgba, int32_t type,
                                                       float exposure) {
    constexpr int h1 = 2 * kCombineRows + 1, h2 = kCombineRows + 1, h3 = kCombineRows / 2 + 1, h4 = kCombineRows / 4 + 1,
                  h5 = kCombineRows / 8 + (kCombineRows < 8 ? 2 : 1);
    __shared__ float u1[33 * h1 * 3], u2[17 * h2 * 3], u3[9 * h3 * 3], u4[5 * h4 * 3], u5[3 * h5 * 3];
    const uint32_t x0 = blockIdx.x * 64, y0 = blockIdx.y * 4 * kCombineRows;
    const uint32_t x = x0 + (threadIdx.x & 63), row = y0 + (threadIdx.x >> 6) * kCombineRows;
    Tile<33, h1> t1;
    Tile<17, h2> t2;
    Tile<9, h3> t3;
    Tile<5, h4> t4;
    Tile<3, h5> t5;
    t5.load(P.level[5], P.dim[5], x0 >> 5, y0 >> 5);
    t4.load(P.level[4], P.dim[4], x0 >> 4, y0 >> 4);
    t3.load(P.level[3], P.dim[3], x0 >> 3, y0 >> 3);
    t2.load(P.level[2], P.dim[2], x0 >> 2, y0 >> 2);
    t1.load(P.level[1], P.dim[1], x0 >> 1, y0 >> 1);
    v3 c[kCombineRows];  // the pixels, read ahead of the walk up the pyramid
#pragma unroll
    for (uint32_t r = 0; r < kCombineRows; ++r)
        c[r] = ld_px(hdr, P.dim[0].w, (int)min(x, P.dim[0].w - 1u), (int)min(row + r, P.dim[0].h - 1u));
    t5.store(u5);
    t4.store(u4);
    t3.store(u3);
    t2.store(u2);
    t1.store(u1);
    __syncthreads();
    gauss_up_tile<5, h4, 3>(u4, x0 >> 4, y0 >> 4, P.dim[4], u5, x0 >> 5, y0 >> 5, P.dim[5]);
    gauss_up_tile<9, h3, 5>(u3, x0 >> 3, y0 >> 3, P.dim[3], u4, x0 >> 4, y0 >> 4, P.dim[4]);
    gauss_up_tile<17, h2, 9>(u2, x0 >> 2, y0 >> 2, P.dim[2], u3, x0 >> 3, y0 >> 3, P.dim[3]);
    gauss_up_tile<33, h1, 17>(u1, x0 >> 1, y0 >> 1, P.dim[1], u2, x0 >> 2, y0 >> 2, P.dim[2]);
    if (x >= P.dim[0].w) return;
    // up(U1) as gauss_up has it, its horizontal means shared by the rows
    const uint32_t cx = (x >> 1) - (x0 >> 1), cx1 = (x & 1u ? min((x >> 1) + 1u, P.dim[1].w - 1u) : x >> 1) - (x0 >> 1);
    const auto mean = [&](uint32_t cy) {
        const float* p = u1 + 3 * 33 * (min(cy, P.dim[1].h - 1u) - (y0 >> 1));
        return (lds_px(p + 3 * cx) + lds_px(p + 3 * cx1)) * 0.5f;
    };
    v3 here = mean(row >> 1), next = here;
#pragma unroll
    for (uint32_t r = 0; r < kCombineRows; ++r) {  // row is even
        const uint32_t y = row + r;
        if (y >= P.dim[0].h) return;
        if (r & 1u)
            next = mean((y >> 1) + 1u);
        else
            here = next;
        const v3 u0 = threshold_px(c[r], curve) + (here + (r & 1u ? next : here)) * 0.5f;
        const v3 o = c[r] + u0 / 6.0f;
        const size_t i = (size_t)y * P.dim[0].w + x;
        st3(out + 3 * i, o);
        if (rgba) rgba[i] = tonemap_px(o, type, exposure);
    }
}

static int gauss_bloom(cupbr_post* p, float4 curve, uint8_t* rgba, int32_t type, float exposure) {
    Pyramid P;
    P.level[0] = nullptr;
    P.dim[0] = {p->width, p->height};
    size_t off[kGaussLevels + 2];
    off[1] = 0;
    for (int k = 1; k <= kGaussLevels; ++k) {
        P.dim[k] = {(P.dim[k - 1].w + 1) / 2, (P.dim[k - 1].h + 1) / 2};
        off[k + 1] = off[k] + (size_t)P.dim[k].w * P.dim[k].h * 3;
    }
    if (int rc = p->levels.ensure(off[kGaussLevels + 1] * sizeof(float))) return rc;
    float* L[kGaussLevels + 1];
    for (int k = 1; k <= kGaussLevels; ++k) P.level[k] = L[k] = p->levels.as<float>() + off[k];
    const auto grid = [&](int k, uint32_t tw, uint32_t th) { return dim3((P.dim[k].w + tw - 1) / tw, (P.dim[k].h + th - 1) / th); };
    hipLaunchKernelGGL(k_gauss_first, grid(1, 32, 8), dim3(256), 0, p->stream, p->hdr, P.dim[0], L[1], P.dim[1], curve);
    hipLaunchKernelGGL(k_gauss_two<8>, grid(3, 8, 8), dim3(256), 0, p->stream, L[1], P.dim[1], L[2], P.dim[2], L[3], P.dim[3]);
    hipLaunchKernelGGL(k_gauss_two<4>, grid(5, 4, 4), dim3(256), 0, p->stream, L[3], P.dim[3], L[4], P.dim[4], L[5], P.dim[5]);
    hipLaunchKernelGGL(k_gauss_combine, grid(0, 64, 4 * kCombineRows), dim3(256), 0, p->stream, p->hdr, P, curve, p->output.as<float>(),
                       reinterpret_cast<uchar4*>(rgba), type, exposure);
    CUPBR_HIP_CHECK(hipGetLastError());
    return CUPBR_OK;
}

int post_bloom(cupbr_post* p, const float curve[4], uint8_t* rgba, int32_t type, float exposure) {
    if (p->width < 2 || p->height < 2)
        return set_error(CUPBR_ERR_INVALID_ARGUMENT, "bloom needs an image of at least 2x2 pixels");
    if (p->pyramid == CUPBR_BLOOM_GAUSSIAN5) {
        CUPBR_HIP_CHECK(hipDeviceSynchronize());  // the registered image is borrowed, as below
        if (int rc = gauss_bloom(p, make_float4(curve[0], curve[1], curve[2], curve[3]), rgba, type, exposure))
            return rc;
        CUPBR_HIP_CHECK(hipStreamSynchronize(p->stream));
        return CUPBR_OK;
    }
    const uint32_t tiles = ((p->width + kTileW - 1) / kTileW) * ((p->height + kTileH - 1) / kTileH);
    dim3 grid(tiles);
    float4 c = make_float4(curve[0], curve[1], curve[2], curve[3]);
    // the registered image is borrowed: finish pending writes to it first, and return only when
    // the outputs are complete (the reference synchronises after every launch, PyramidConstructor.cu:134)
    CUPBR_HIP_CHECK(hipDeviceSynchronize());
    hipLaunchKernelGGL(k_bloom, grid, dim3(256), 0, p->stream, p->hdr, p->output.as<float>(),
                       reinterpret_cast<uchar4*>(rgba), p->width, p->height, c, type, exposure);
    CUPBR_HIP_CHECK(hipGetLastError());
    CUPBR_HIP_CHECK(hipStreamSynchronize(p->stream));
    return CUPBR_OK;
}

int tonemap(cupbr_tonemapper* t) {
    const size_t n = (size_t)t->width * t->height;
    CUPBR_HIP_CHECK(hipDeviceSynchronize());
    hipLaunchKernelGGL(k_tonemap, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, t->stream, t->hdr,
                       t->rgba.as<uchar4>(), n, t->type, t->exposure);
    CUPBR_HIP_CHECK(hipGetLastError());
    CUPBR_HIP_CHECK(hipStreamSynchronize(t->stream));  // ToneMapper.cu:172
    return CUPBR_OK;
}

// The bytes of every float by power_byte and by powf for the three power curves, and Reinhard's base in float and in
// double for every exponential: counts of those that differ.
__global__ __launch_bounds__(256) void k_tone_byte_check(unsigned long long* differing) {
    uint32_t n[4] = {0, 0, 0, 0};
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < (1ull << 32); i += stride) {
        const float x = __uint_as_float((uint32_t)i);
        const float g0 = 1.0f / 2.2f, g1 = (float)(1.0f / 2.2), g2 = 1.0f / 2.4f;
        n[0] += power_byte(x, g0, 1.0f, 0.0f) != to_byte(powf(x, g0)) ? 1u : 0u;
        n[1] += power_byte(x, g1, 1.0f, 0.0f) != to_byte(powf(x, g1)) ? 1u : 0u;
        if (!(x <= 0.0031308f)) n[2] += power_byte(x, g2, 1.055f, -0.055f) != to_byte(1.055f * powf(x, g2) - 0.055f) ? 1u : 0u;
        const float a = 1.0f - x, b = (float)(1.0 - (double)x);
        n[3] += __float_as_uint(a) != __float_as_uint(b) && (a == a || b == b) ? 1u : 0u;
    }
    for (int k = 0; k < 4; ++k) {
        for (int off = 32; off > 0; off >>= 1) n[k] += __shfl_xor(n[k], off);
        if (__lane_id() == 0 && n[k]) atomicAdd(differing + k, (unsigned long long)n[k]);
    }
}

int tone_byte_check(uint64_t differing[4]) {
    DevBuf d;
    if (int rc = d.ensure(4 * sizeof(uint64_t))) return rc;
    CUPBR_HIP_CHECK(hipMemset(d.ptr, 0, 4 * sizeof(uint64_t)));
    hipLaunchKernelGGL(k_tone_byte_check, dim3(device_cu_count() * 8), dim3(256), 0, nullptr, d.as<unsigned long long>());
    CUPBR_HIP_CHECK(hipGetLastError());
    CUPBR_HIP_CHECK(hipMemcpy(differing, d.ptr, 4 * sizeof(uint64_t), hipMemcpyDeviceToHost));
    return CUPBR_OK;
}

// 32-bit BI_RGB bitmap, bottom-up: buffer row 0 is written first and shown at the bottom,
// as stbi_write_bmp does after stbi_flip_vertically_on_write(true) (ToneMapper.cu:194-195)
int write_bmp(const char* path, const uint8_t* rgba, uint32_t w, uint32_t h) {
    FILE* f = fopen(path, "wb");
    if (!f) return set_error(CUPBR_ERR_FILE, std::string("cannot write ") + path, true);
    const uint32_t data = w * h * 4, off = 14 + 40, size = off + data;
    uint8_t hdr[54] = {'B', 'M'};
    auto put32 = [&](int at, uint32_t v) { for (int k = 0; k < 4; ++k) hdr[at + k] = (uint8_t)(v >> (8 * k)); };
    put32(2, size);
    put32(10, off);
    put32(14, 40);
    put32(18, w);
    put32(22, h);
    hdr[26] = 1;
    hdr[28] = 32;
    put32(34, data);
    put32(38, 2835);
    put32(42, 2835);
    bool ok = fwrite(hdr, 1, 54, f) == 54;
    std::vector<uint8_t> row((size_t)w * 4);
    for (uint32_t y = 0; y < h && ok; ++y) {
        for (uint32_t x = 0; x < w; ++x) {
            const uint8_t* s = rgba + 4 * ((size_t)y * w + x);
            row[4 * x] = s[2];
            row[4 * x + 1] = s[1];
            row[4 * x + 2] = s[0];
            row[4 * x + 3] = s[3];
        }
        ok = fwrite(row.data(), 1, row.size(), f) == row.size();
    }
    fclose(f);
    return ok ? CUPBR_OK : set_error(CUPBR_ERR_FILE, std::string("write failed: ") + path, true);
}

}  // namespace cupbr
