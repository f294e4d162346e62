// Neural radiance cache: a 64 -> 64 -> 64 -> 64 -> 64 -> 3 ReLU MLP without biases (16,576
// weights), BF16 operands on the CDNA4 matrix cores (v_mfma_f32_16x16x32_bf16) with FP32
// accumulation, trained online with Adam on a relative L2 loss. No counterpart in the reference.
//
// Inputs (16 floats per query): position (3, world), outgoing direction wo (3, unit), shading
// normal (3, unit), roughness (1), diffuse albedo (3), specular albedo (3). Encoding (64 features):
//   0..35   sin/cos(2^k pi p_a), p normalised to the cache's box, a = 0..2, k = 0..5
//   36..43  sin/cos(2^k pi x), x = acos(wo.z)/pi and (atan2(wo.y, wo.x)/pi + 1)/2, k = 0..1
//   44..51  the same for the normal
//   52      1 - exp(-roughness);  53..55 diffuse albedo;  56..58 specular albedo;  59 one; 60..63 zero
//
// Matrix-core layout (one wave, 16 queries per tile; queries are the N dimension):
//   D[16 x 16] += A[16 x 32] * B[32 x 16]; lane l holds A[l%16][8(l/16) + j], B[8(l/16) + j][l%16]
//   (j = 0..7) and D[4(l/16) + v][l%16] (v = 0..3).
// A layer's 64 outputs are 4 D tiles; lane l then holds outputs t*16 + 4(l/16) + v of query l%16,
// t = 0..3. Those 16 values become the next layer's B operand unchanged: K slot kk of chunk kc
// stands for feature perm(kc, kk) = (2kc + (kk%8)/4)*16 + (kk/8)*4 + kk%4, and the weights are
// stored pre-permuted to match, so activations never leave registers between layers.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "device.h"
#include "nrc.h"

namespace cupbr {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kFwdLayer = 4096;                           // bf16 per packed 64x64 layer
constexpr int kFwdSize = 4 * kFwdLayer + 2 * 64 * 8;      // + W5 (one output tile)
constexpr int kBwdSize = 3 * kFwdLayer + 4 * 64 * 8;      // W2^T..W4^T + W5^T
constexpr int kNrcBlock = 256;

__device__ __forceinline__ __bf16 to_bf16(float x) { return (__bf16)x; }

// max(x, 0) before the rounding to BF16, 0 for a NaN, in one instruction (fmaxf of a matrix-core result
// takes two: it first quietens a signalling NaN). The upper end only keeps the compiler from turning
// this into that fmaxf: the largest float rounds to infinity in BF16, as infinity does.
__device__ __forceinline__ float relu(float x) { return __builtin_amdgcn_fmed3f(x, 0.0f, 3.402823466e38f); }

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// sin(pi y) and cos(pi y) from the hardware's sine and cosine, whose argument is in revolutions
// (v_sin_f32(r) = sin(2 pi r)): r = y / 2 is exact, and its fraction keeps the argument in [0, 1),
// well inside the instructions' input range. Their error (~1e-6 absolute) is far below the BF16
// rounding the feature then takes.
__device__ __forceinline__ void sincospi_hw(float y, float* s, float* c) {
    float r = 0.5f * y;
    r -= floorf(r);
    *s = __builtin_amdgcn_sinf(r);
    *c = __builtin_amdgcn_cosf(r);
}

// the four features sin, cos(pi y), sin, cos(2 pi y)
__device__ __forceinline__ void octaves(float y, float f[4]) {
    sincospi_hw(y, &f[0], &f[1]);
    sincospi_hw(2.0f * y, &f[2], &f[3]);
}

// B operand of the first layer for lane group g: slot (kc, j) holds feature perm(kc, 8g + j), that is,
// output tile t = 2kc + j/4 of a layer holds features 16t + 4g .. 16t + 4g + 3. A lane computes its own
// 16 features only: two octaves of one coordinate per tile (their arguments 2^k x are exact), and of
// the four angles the one that its group needs (g = 1: acos(wo.z), 2: atan2(wo), 3: acos(n.z), 0:
// atan2(n)), so that a query costs one acos and one atan2 per lane, not four.
__device__ __forceinline__ void encode(const NrcBox& box, const float* raw, int g, bf16x8 b[2]) {
    const float pi = 3.14159265358979f;
    float x[3];
    for (int a = 0; a < 3; ++a) x[a] = (raw[a] - box.lo[a]) * box.inv_ext[a];
    const float polar = acosf(fminf(fmaxf(g == 1 ? raw[5] : raw[8], -1.0f), 1.0f)) / pi;
    const float azimuth = (atan2f(g == 2 ? raw[4] : raw[7], g == 2 ? raw[3] : raw[6]) / pi + 1.0f) * 0.5f;
    const float angle = (g & 1) ? polar : azimuth;
    float f[4][4];
    // features 0..35 are (x, y, z) x octaves 0..5: tile 0 holds x 0-1, x 2-3, x 4-5, y 0-1 for g = 0..3,
    // tile 1 y 2-3, y 4-5, z 0-1, z 2-3, tile 2 z 4-5 (g = 0)
    octaves((g == 3 ? x[1] : x[0]) * (g == 1 ? 4.0f : g == 2 ? 16.0f : 1.0f), f[0]);
    octaves((g < 2 ? x[1] : x[2]) * (g == 1 ? 16.0f : g == 2 ? 1.0f : 4.0f), f[1]);
    octaves(g == 0 ? x[2] * 16.0f : angle, f[2]);
    octaves(angle, f[3]);
    if (g != 0) {  // roughness, albedos, one, zeros
        f[3][0] = g == 1 ? 1.0f - expf(-raw[9]) : g == 2 ? raw[13] : 0.0f;
        f[3][1] = g == 1 ? raw[10] : g == 2 ? raw[14] : 0.0f;
        f[3][2] = g == 1 ? raw[11] : g == 2 ? raw[15] : 0.0f;
        f[3][3] = g == 1 ? raw[12] : g == 2 ? 1.0f : 0.0f;
    }
    for (int kc = 0; kc < 2; ++kc)
        for (int j = 0; j < 8; ++j) b[kc][j] = to_bf16(f[2 * kc + (j >> 2)][j & 3]);
}

// one hidden layer: out = relu(W x) as the next B operand; w = packed fragments [ot][kc][lane][8]
__device__ __forceinline__ void hidden_layer(const bf16x8* w, int lane, const bf16x8 in[2], bf16x8 out[2],
                                             f32x4* pre = nullptr) {
    f32x4 acc[4];
    for (int ot = 0; ot < 4; ++ot) {
        acc[ot] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int kc = 0; kc < 2; ++kc) acc[ot] = mfma(w[(ot * 2 + kc) * 64 + lane], in[kc], acc[ot]);
    }
    for (int kc = 0; kc < 2; ++kc)
        for (int j = 0; j < 8; ++j) out[kc][j] = to_bf16(relu(acc[2 * kc + (j >> 2)][j & 3]));
    if (pre)
        for (int ot = 0; ot < 4; ++ot) pre[ot] = acc[ot];
}

// hidden_layer for two tiles of 16 queries, its 8 weight fragments in registers
__device__ __forceinline__ void hidden_layer2(const bf16x8* w, const bf16x8 in0[2], const bf16x8 in1[2],
                                              bf16x8 out0[2], bf16x8 out1[2]) {
    f32x4 acc0[4], acc1[4];
#pragma unroll
    for (int ot = 0; ot < 4; ++ot) {
        acc0[ot] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        acc1[ot] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int kc = 0; kc < 2; ++kc) {
            acc0[ot] = mfma(w[ot * 2 + kc], in0[kc], acc0[ot]);
            acc1[ot] = mfma(w[ot * 2 + kc], in1[kc], acc1[ot]);
        }
    }
#pragma unroll
    for (int kc = 0; kc < 2; ++kc)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            out0[kc][j] = to_bf16(relu(acc0[2 * kc + (j >> 2)][j & 3]));
            out1[kc][j] = to_bf16(relu(acc1[2 * kc + (j >> 2)][j & 3]));
        }
}

// output layer: lane group 0 gets the 3 outputs (v = 0..2) of query lane%16
__device__ __forceinline__ f32x4 output_layer(const bf16x8* w5, int lane, const bf16x8 in[2]) {
    f32x4 acc{0.0f, 0.0f, 0.0f, 0.0f};
    for (int kc = 0; kc < 2; ++kc) acc = mfma(w5[kc * 64 + lane], in[kc], acc);
    return acc;
}

// inference over n queries of `stride` floats (first 16 = inputs). kAccumulate: out_rgb[path] +=
// thr * max(pred, 0) with thr = record[16..18] and path = bits of record[19]; else out[q*3 + c] = pred.
//
// Bound by VALU issue (the encoding and the ReLU and rounding between the layers, some 800 instructions
// per 32 queries and lane, beside 68 matrix instructions). Every wave keeps the whole network's 34
// weight fragments in registers (136 of its 256: 2 waves per SIMD) and runs through the queries, two
// tiles of 16 at a time; read from LDS they were 34 KB per 32 queries, as long as the matrix
// instructions themselves. 1,000,003 queries: 97.7 us with the weights in LDS and every lane encoding
// all four angles, 61.4 with both changed, 54.3 (610 TFLOP/s) with the one-instruction relu.
template <bool kAccumulate>
__global__ __launch_bounds__(kNrcBlock, 2) void k_nrc_infer(const bf16x8* __restrict__ packed, NrcBox box,
                                                            const float* __restrict__ rec, uint32_t n,
                                                            const uint32_t* __restrict__ n_dev, uint32_t stride,
                                                            float* __restrict__ out,
                                                            const uint32_t* __restrict__ begin_dev, NrcParts parts) {
    const int lane = threadIdx.x & 63, g = lane >> 4;
    bf16x8 w[kFwdSize / 512];  // loaded while the counts are
#pragma unroll
    for (int i = 0; i < kFwdSize / 512; ++i) w[i] = packed[i * 64 + lane];
    uint32_t blk = blockIdx.x, blks = gridDim.x, begin = 0;
    if (kAccumulate && parts.size != 0u) {  // an XCD's part by its own blocks
        const uint32_t x = blk & 7u;
        blk >>= 3;
        blks >>= 3;
        begin = x * parts.size;
        n = begin + min(parts.size, n_dev[x * parts.stride]);
    } else {
        if (n_dev) n = min(n, *n_dev);  // count written by an earlier kernel on the stream
        begin = begin_dev ? min(*begin_dev, n) : 0u;
    }
    const uint32_t wave = (blk * blockDim.x + threadIdx.x) >> 6;
    const uint32_t n_waves = (blks * blockDim.x) >> 6;
    const uint32_t pairs = (n - begin + 31) / 32;  // two tiles of 16 queries per wave and step
    if (wave >= pairs) return;
    for (uint32_t t = wave; t < pairs; t += n_waves) {
        uint32_t q[2];
        bf16x8 a[2][2], b[2][2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            q[h] = begin + t * 32 + 16 * h + (lane & 15);
            float raw[16];
            if (q[h] < n) {
                const float4* r4 = reinterpret_cast<const float4*>(rec + (size_t)q[h] * stride);
                for (int k = 0; k < 4; ++k) {
                    const float4 v = r4[k];
                    raw[4 * k] = v.x;
                    raw[4 * k + 1] = v.y;
                    raw[4 * k + 2] = v.z;
                    raw[4 * k + 3] = v.w;
                }
            } else {
                for (int k = 0; k < 16; ++k) raw[k] = 0.0f;
                raw[5] = 1.0f;
                raw[8] = 1.0f;
            }
            encode(box, raw, g, a[h]);
        }
        // the path's throughput and radiance while the layers run
        f32x4 thr[2];
        float* px[2];
        float rgb[2][3];
        if (kAccumulate && g == 0) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (q[h] >= n) continue;
                const float* r = rec + (size_t)q[h] * stride;
                thr[h] = f32x4{r[16], r[17], r[18], r[19]};
                px[h] = out + 4 * (size_t)__float_as_uint(thr[h][3]);
                for (int k = 0; k < 3; ++k) rgb[h][k] = px[h][k];
            }
        }
        hidden_layer2(w, a[0], a[1], b[0], b[1]);
        hidden_layer2(w + 8, b[0], b[1], a[0], a[1]);
        hidden_layer2(w + 16, a[0], a[1], b[0], b[1]);
        hidden_layer2(w + 24, b[0], b[1], a[0], a[1]);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            f32x4 o{0.0f, 0.0f, 0.0f, 0.0f};  // lane group 0 gets the 3 outputs of query lane % 16
            for (int kc = 0; kc < 2; ++kc) o = mfma(w[32 + kc], a[h][kc], o);
            if (g == 0 && q[h] < n) {
                if (kAccumulate) {
                    for (int k = 0; k < 3; ++k) px[h][k] = rgb[h][k] + thr[h][k] * fmaxf(o[k], 0.0f);
                } else {
                    out[3 * (size_t)q[h] + 0] = o[0];
                    out[3 * (size_t)q[h] + 1] = o[1];
                    out[3 * (size_t)q[h] + 2] = o[2];
                }
            }
        }
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

// Training state on the device: steps taken since the weights were set, and the number of the step at
// hand (each written by one thread of a launch that does not read it).
struct TrainState {
    uint32_t taken, step;
};

// Step s of a call: forward, loss and backward for one training batch of B rows (a multiple of 64), 64
// rows per tile. Batch row q is rows[hash(seed + q) % n_rows], its seed from the step number.
//
// A wave takes 16 rows through the network in registers (the weights of both directions in LDS). The
// weight gradients dW[o][i] = sum_q G[o][q] X[i][q] of k_nrc_weight_sums then need the batch rows as the K
// dimension: the inputs X of the five layers and the loss gradients G at their outputs go through LDS
// as [feature][row] (rows of 64 + 8 values, so that the 16 lanes of an operand load read all 64 banks
// once) and from there to memory as matrix operands, acts[row / 512][operand][row % 512 / 32][lane] of 16
// bytes: operands 0..19 are X[layer][16 features], 20..35 G[hidden layer][16 outputs], 36 the output
// layer's G.
// Bound by the latency of one 16-row chain per SIMD and the 20 MB of operands. 16,384 rows: 26.7 us when
// every value went to memory as a 2-byte store and the weights to LDS one load after the other, now
// 11.3; 16.7 with operands 16 KB apart, 14.6 with a slice's tiles on all XCDs.
constexpr int kTrainRows = 64;
constexpr int kTrainStride = kTrainRows + 8;
constexpr uint32_t kOperands = 37;
constexpr uint32_t kSlice = 512;                         // batch rows whose gradients are added up first
// 16-byte values of one operand of a slice, and 1 KB between operands: 16 KB apart, the pieces that a
// block writes of every operand would share memory channels
constexpr uint32_t kSliceOperand = kSlice / 32 * 64 + 64;
constexpr uint32_t kSliceTiles = kSlice / kTrainRows;
// The u-th tile of a batch: a slice's tiles are 8 apart, so that (blocks going round the XCDs) one XCD
// makes all of a slice, the one on which k_nrc_weight_sums reads it.
__device__ __forceinline__ uint32_t tile_at(uint32_t u) {
    return ((u / (8u * kSliceTiles)) * 8u + (u & 7u)) * kSliceTiles + (u >> 3) % kSliceTiles;
}

__device__ __forceinline__ void store_rows(__bf16* base, int row, int g, const bf16x8 v[2]) {
#pragma unroll
    for (int kc = 0; kc < 2; ++kc)
#pragma unroll
        for (int j = 0; j < 8; ++j) base[((2 * kc + (j >> 2)) * 16 + g * 4 + (j & 3)) * kTrainStride + row] = v[kc][j];
}

__global__ __launch_bounds__(kNrcBlock, 1) void k_nrc_train(const bf16x8* __restrict__ pf, const bf16x8* __restrict__ pb,
                                                            NrcBox box, const float* __restrict__ rows, uint32_t n_rows,
                                                            const uint32_t* __restrict__ n_rows_dev, uint32_t B,
                                                            TrainState* state, uint32_t s, bf16x8* __restrict__ acts,
                                                            float* __restrict__ losses) {
    __shared__ bf16x8 wf[kFwdSize / 8];
    __shared__ bf16x8 wb[kBwdSize / 8];
    // [feature][row], 16 features per operand: X of the 5 layers, G of the 4 hidden ones, G of the output layer
    __shared__ __attribute__((aligned(16))) __bf16 xg[kOperands * 16 * kTrainStride];
    __bf16* const g5 = xg + 36 * 16 * kTrainStride;
    __shared__ float loss_s[kNrcBlock / 64];
    const int lane = threadIdx.x & 63, g = lane >> 4, wave = threadIdx.x >> 6;
    const int col = wave * 16 + (lane & 15);
    // the weights, the counts and then the first row: their loads in flight together (the weights one
    // after the other take 7 us more)
    constexpr int nf = (kFwdSize / 8 + kNrcBlock - 1) / kNrcBlock, nb = (kBwdSize / 8 + kNrcBlock - 1) / kNrcBlock;
    bf16x8 f[nf], b[nb];
#pragma unroll
    for (int k = 0; k < nf; ++k) f[k] = pf[min((int)threadIdx.x + k * kNrcBlock, kFwdSize / 8 - 1)];
#pragma unroll
    for (int k = 0; k < nb; ++k) b[k] = pb[min((int)threadIdx.x + k * kNrcBlock, kBwdSize / 8 - 1)];
    if (n_rows_dev) n_rows = min(n_rows, *n_rows_dev);
    const uint32_t step = state->taken + s + 1u;
    if (n_rows == 0) return;
    if (tile_at(blockIdx.x) >= B / kTrainRows) {  // the last slices of a batch that is no multiple of 4096 rows
        if (threadIdx.x == 0) losses[blockIdx.x] = 0.0f;
        return;
    }
    const uint32_t seed = step * 0x9E3779B9u + 0x51ED270Bu;
    float raw[19];
    auto load_row = [&](uint32_t t) {
        const float* r = rows + (size_t)(hash32(seed + t * kTrainRows + col) % n_rows) * kNrcRowStride;
#pragma unroll
        for (int k = 0; k < 19; ++k) raw[k] = r[k];
    };
    load_row(tile_at(blockIdx.x));
    bf16x8 x[5][2];
    encode(box, raw, g, x[0]);  // while the weights arrive
#pragma unroll
    for (int k = 0; k < nf; ++k)
        if ((int)threadIdx.x + k * kNrcBlock < kFwdSize / 8) wf[threadIdx.x + k * kNrcBlock] = f[k];
#pragma unroll
    for (int k = 0; k < nb; ++k)
        if ((int)threadIdx.x + k * kNrcBlock < kBwdSize / 8) wb[threadIdx.x + k * kNrcBlock] = b[k];
    __syncthreads();
    float loss_acc = 0.0f;
    for (uint32_t u = blockIdx.x; tile_at(u) < B / kTrainRows; u += gridDim.x) {  // gridDim.x: a multiple of 64
        const uint32_t t = tile_at(u);
        if (u != blockIdx.x) {
            load_row(t);
            encode(box, raw, g, x[0]);
        }
        f32x4 pre[4][4];
#pragma unroll
        for (int L = 0; L < 4; ++L) hidden_layer(wf + L * (kFwdLayer / 8), lane, x[L], x[L + 1], pre[L]);
        const f32x4 o = output_layer(wf + 4 * (kFwdLayer / 8), lane, x[4]);
        // relative L2: sum_c (o_c - y_c)^2 / (o_c^2 + 0.01), o_c detached in the denominator
        bf16x8 cur[2];
#pragma unroll
        for (int kc = 0; kc < 2; ++kc)
#pragma unroll
            for (int j = 0; j < 8; ++j) cur[kc][j] = to_bf16(0.0f);
        if (g == 0) {
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const float den = o[c] * o[c] + 0.01f;
                const float e = o[c] - raw[16 + c];
                loss_acc += e * e / den;
                cur[0][c] = to_bf16(2.0f * e / den);
            }
        }
#pragma unroll
        for (int L = 0; L < 5; ++L) store_rows(xg + L * 64 * kTrainStride, col, g, x[L]);
#pragma unroll
        for (int j = 0; j < 4; ++j) g5[(g * 4 + j) * kTrainStride + col] = g == 0 ? cur[0][j] : to_bf16(0.0f);
        // backward through W5^T, then W4^T..W2^T, masking with the ReLU of each hidden layer
#pragma unroll
        for (int L = 3; L >= 0; --L) {
            f32x4 acc[4];
#pragma unroll
            for (int it = 0; it < 4; ++it) {
                acc[it] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                if (L == 3) {
                    acc[it] = mfma(wb[3 * (kFwdLayer / 8) + it * 64 + lane], cur[0], acc[it]);
                } else {
#pragma unroll
                    for (int kc = 0; kc < 2; ++kc)
                        acc[it] = mfma(wb[L * (kFwdLayer / 8) + (it * 2 + kc) * 64 + lane], cur[kc], acc[it]);
                }
            }
#pragma unroll
            for (int kc = 0; kc < 2; ++kc)
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int ot = 2 * kc + (j >> 2), v = j & 3;
                    cur[kc][j] = to_bf16(pre[L][ot][v] > 0.0f ? acc[ot][v] : 0.0f);
                }
            store_rows(xg + (5 + L) * 64 * kTrainStride, col, g, cur);
        }
        __syncthreads();
        // operand rows: lane l holds row l % 16 of its 16 features, batch rows 32 half + 8 (l / 16) .. + 7.
        // Wave w copies half w % 2 of operands w / 2, w / 2 + 2, .., all reads in flight together (a step of 4096
        // rows 15.3 -> 13.9 us)
        const uint32_t half = wave & 1u, op0 = wave >> 1;
        const __bf16* from = xg + (op0 * 16u + (lane & 15u)) * kTrainStride + 32u * half + 8u * g;
        bf16x8* to = acts + ((size_t)(t / kSliceTiles) * kOperands + op0) * kSliceOperand +
                     t % kSliceTiles * (kTrainRows / 32 * 64) + half * 64u + lane;
        constexpr uint32_t n_copies = (kOperands + 1) / 2;
        bf16x8 v[n_copies];
#pragma unroll
        for (uint32_t j = 0; j < n_copies; ++j)
            if (op0 + 2u * j < kOperands) v[j] = *reinterpret_cast<const bf16x8*>(from + j * 32u * kTrainStride);
#pragma unroll
        for (uint32_t j = 0; j < n_copies; ++j)
            if (op0 + 2u * j < kOperands) to[j * 2u * kSliceOperand] = v[j];
        __syncthreads();
    }
    for (int off = 32; off > 0; off >>= 1) loss_acc += __shfl_xor(loss_acc, off);
    if (lane == 0) loss_s[wave] = loss_acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        float sum = 0.0f;
        for (int k = 0; k < kNrcBlock / 64; ++k) sum += loss_s[k];
        losses[blockIdx.x] = sum;
        if (blockIdx.x == 0) state->step = step;
    }
}

__device__ __forceinline__ void pack_weight(uint32_t p, float w, __bf16* __restrict__ pf, __bf16* __restrict__ pb);

// Weight gradients of slices of 512 batch rows: one wave takes a slice of one 16 x 16 tile of a layer's
// weights through 16 matrix instructions in row order, all 32 operand loads in flight together. The
// order of the rows, and of the slices in k_nrc_adam, is fixed: it decides the last bits of the gradients,
// and with them when a BF16 weight or a ReLU tips over in later steps.
// A block holds the four tiles of 16 outputs of a layer, which share the G operand; the 17 blocks of a
// slice run on one XCD (ids 8 apart), so that its 629 KB of operands reach one L2. Bound by the latency of
// those loads (16,384 rows: 5.1 us; 10.7 with a slice's tiles on all XCDs; 12.1 in 160 waves that took all
// 16 tiles of a layer through their chunks one load after the other).
// sums[tile][slice][lane]: lane 16 a + i holds outputs 4 a .. 4 a + 3 of input i.
constexpr uint32_t kWeightTiles = 68;  // 4 layers of 4 x 4, and 4 of the output layer
__global__ __launch_bounds__(kNrcBlock) __attribute__((amdgpu_waves_per_eu(1, 3)))
void k_nrc_weight_sums(const bf16x8* __restrict__ acts, uint32_t n_slices, f32x4* __restrict__ sums, uint32_t n_rows,
                       const uint32_t* __restrict__ n_rows_dev) {
    if (n_rows_dev && min(n_rows, *n_rows_dev) == 0u) return;
    const int lane = threadIdx.x & 63;
    const uint32_t r = blockIdx.x >> 3, s = r / 17u * 8u + (blockIdx.x & 7u), L = r % 17u >> 2, ot = r % 17u & 3u;
    if (s >= n_slices) return;
    const uint32_t it = threadIdx.x >> 6, tile = L * 16u + ot * 4u + it;  // L = 4, ot = 0: the output layer
    const bf16x8* base = acts + (size_t)s * kOperands * kSliceOperand + lane;
    const bf16x8* ga = base + (20u + L * 4u + ot) * kSliceOperand;
    const bf16x8* xa = base + (L * 4u + it) * kSliceOperand;
    bf16x8 a[kSlice / 32], x[kSlice / 32];
#pragma unroll
    for (uint32_t k = 0; k < kSlice / 32; ++k) {
        a[k] = ga[k * 64u];
        x[k] = xa[k * 64u];
    }
    f32x4 acc{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (uint32_t k = 0; k < kSlice / 32; ++k) acc = mfma(a[k], x[k], acc);
    sums[((size_t)tile * n_slices + s) * 64 + lane] = acc;
}

// The sum of the slices in order, Adam, and the packed BF16 copies for the next batch: a block per
// weight tile (thread 64 a + 4 i + v: output 4 a + v, input i), and one that adds up the loss. Bound by
// latency: the loads of up to 32 slices are in flight together (16,384 rows: 9.8 us with one load and add
// after the other, now 3.6).
constexpr uint32_t kBiasSteps = 2048;  // from here on 1 - beta^t is 1 in FP32
__global__ __launch_bounds__(kNrcBlock) void k_nrc_adam(const f32x4* __restrict__ sums, uint32_t n_slices,
                                                        const float* __restrict__ losses, uint32_t n_losses, float inv_b,
                                                        float* __restrict__ w, float* __restrict__ m,
                                                        float* __restrict__ v, float lr, float b1, float b2, float eps,
                                                        const float2* __restrict__ bias, uint32_t n_rows,
                                                        const uint32_t* __restrict__ n_rows_dev, TrainState* state,
                                                        uint32_t add_taken, float* loss, __bf16* __restrict__ pf,
                                                        __bf16* __restrict__ pb) {
    const uint32_t tile = blockIdx.x;
    if (n_rows_dev && min(n_rows, *n_rows_dev) == 0u) return;
    if (tile == kWeightTiles) {
        const uint32_t lane = threadIdx.x;
        if (lane >= 64u) return;
        float sum = 0.0f;
        for (uint32_t k = lane; k < n_losses; k += 64) sum += losses[k];
        for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
        if (lane == 0) {
            if (loss) *loss += sum;
            state->taken += add_taken;  // after the call's last batch: no launch in flight reads it
        }
        return;
    }
    const uint32_t a = threadIdx.x >> 6, i = (threadIdx.x >> 2) & 15u, k4 = threadIdx.x & 3u;
    const uint32_t o = (tile < 64u ? (tile >> 2) & 3u : 0u) * 16u + a * 4u + k4;
    if (tile >= 64u && o >= 3u) return;
    const uint32_t p = (tile >> 4) * 4096u + o * 64u + (tile & 3u) * 16u + i;
    const float* mine = reinterpret_cast<const float*>(sums + (size_t)tile * n_slices * 64 + a * 16u + i) + k4;
    const float m0 = m[p], v0 = v[p], w0 = w[p];
    const float2 bc = bias[min(state->step, kBiasSteps - 1u)];
    float gsum = 0.0f;
    for (uint32_t s = 0; s < n_slices; s += 32) {
        float q[32];
#pragma unroll
        for (uint32_t k = 0; k < 32; ++k) q[k] = mine[(size_t)min(s + k, n_slices - 1u) * 256];
#pragma unroll
        for (uint32_t k = 0; k < 32; ++k)
            if (s + k < n_slices) gsum += q[k];
    }
    const float gr = gsum * inv_b;
    const float mm = b1 * m0 + (1.0f - b1) * gr;
    const float vv = b2 * v0 + (1.0f - b2) * gr * gr;
    m[p] = mm;
    v[p] = vv;
    const float wn = w0 - lr * (mm / bc.x) / (sqrtf(vv / bc.y) + eps);
    w[p] = wn;
    pack_weight(p, wn, pf, pb);
}

// the BF16 copies of parameter p = weight W_L[o][i] at its fragment positions (see the file
// comment) in the forward and backward layouts
__device__ __forceinline__ void pack_weight(uint32_t p, float w, __bf16* __restrict__ pf, __bf16* __restrict__ pb) {
    const int L = p < 4 * 4096 ? (int)(p / 4096) : 4;
    const int local = L < 4 ? (int)(p % 4096) : (int)(p - 4 * 4096);
    const int o = local / 64, i = local % 64;
    const __bf16 val = (__bf16)w;
    // forward: A[o][k] with k -> input i
    {
        const int t = i / 16, g = (i % 16) / 4, vv = i % 4, kc = t / 2, j = (t % 2) * 4 + vv;
        const int lane = g * 16 + o % 16, ot = o / 16;
        pf[L * 4096 + ((ot * 2 + kc) * 64 + lane) * 8 + j] = val;
    }
    // backward: A[i][k] with k -> output o (layers 2..5 only)
    if (L >= 1) {
        const int it = i / 16;
        if (L < 4) {
            const int t = o / 16, g = (o % 16) / 4, vv = o % 4, kc = t / 2, j = (t % 2) * 4 + vv;
            const int lane = g * 16 + i % 16;
            pb[(L - 1) * 4096 + ((it * 2 + kc) * 64 + lane) * 8 + j] = val;
        } else {
            const int lane = i % 16, j = o;  // o < 3: group 0, slot o
            pb[3 * 4096 + (it * 64 + lane) * 8 + j] = val;
        }
    }
}

__global__ void k_nrc_pack(const float* __restrict__ w, __bf16* __restrict__ pf, __bf16* __restrict__ pb) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < kNrcParams) pack_weight(p, w[p], pf, pb);
}

// D = A * B through one matrix-core instruction with the fragment layout above (A 16x32, B 32x16,
// row-major FP32 in, rounded to BF16): the self-check of that layout
__global__ __launch_bounds__(64) void k_nrc_mfma_product(const float* __restrict__ a, const float* __restrict__ b,
                                                         float* __restrict__ d) {
    const int lane = threadIdx.x, g = lane >> 4, r = lane & 15;
    bf16x8 fa, fb;
    for (int j = 0; j < 8; ++j) {
        fa[j] = to_bf16(a[r * 32 + 8 * g + j]);
        fb[j] = to_bf16(b[(8 * g + j) * 16 + r]);
    }
    const f32x4 acc = mfma(fa, fb, f32x4{0.0f, 0.0f, 0.0f, 0.0f});
    for (int v = 0; v < 4; ++v) d[(4 * g + v) * 16 + r] = acc[v];
}

}  // namespace cupbr

using namespace cupbr;

// ------------------------------------------------------------------ host side
static uint64_t splitmix(uint64_t& s) {
    uint64_t z = (s += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

namespace cupbr {

int nrc_init_weights(cupbr_nrc* c, uint32_t seed) {
    // He-normal hidden layers (std sqrt(2/64)), output layer std 0.01
    std::vector<float> w(kNrcParams);
    uint64_t s = 0x1234ABCDull ^ ((uint64_t)seed << 32);
    for (uint32_t p = 0; p < kNrcParams; p += 2) {
        const double u1 = ((splitmix(s) >> 11) + 0.5) * (1.0 / 9007199254740992.0);
        const double u2 = ((splitmix(s) >> 11) + 0.5) * (1.0 / 9007199254740992.0);
        const double r = std::sqrt(-2.0 * std::log(u1)), a = 2.0 * 3.14159265358979323846 * u2;
        const double n0 = r * std::cos(a), n1 = r * std::sin(a);
        for (int k = 0; k < 2 && p + k < kNrcParams; ++k) {
            const uint32_t q = p + k;
            const double sd = q < 4 * 4096 ? std::sqrt(2.0 / 64.0) : 0.01;
            w[q] = (float)((k ? n1 : n0) * sd);
        }
    }
    return nrc_set_weights(c, w.data());
}

int nrc_set_weights(cupbr_nrc* c, const float* host) {
    CUPBR_HIP_CHECK(hipMemcpy(c->w.ptr, host, kNrcParams * 4, hipMemcpyHostToDevice));
    CUPBR_HIP_CHECK(hipMemset(c->moments.ptr, 0, 2 * kNrcParams * 4 + sizeof(TrainState)));
    return nrc_pack(c, nullptr);
}

int nrc_pack(cupbr_nrc* c, hipStream_t stream) {
    hipLaunchKernelGGL(k_nrc_pack, dim3((kNrcParams + 255) / 256), dim3(256), 0, stream, c->w.as<float>(),
                       c->packed_fwd.as<__bf16>(), c->packed_bwd.as<__bf16>());
    CUPBR_HIP_CHECK(hipGetLastError());
    return CUPBR_OK;
}

int nrc_create(const float lo[3], const float hi[3], uint32_t seed, cupbr_nrc** out) {
    auto* c = new cupbr_nrc();
    for (int a = 0; a < 3; ++a) {
        c->box.lo[a] = lo[a];
        const float e = hi[a] - lo[a];
        c->box.inv_ext[a] = e > 0.0f ? 1.0f / e : 1.0f;
    }
    int rc;
    if ((rc = c->w.ensure(kNrcParams * 4)) || (rc = c->moments.ensure(2 * kNrcParams * 4 + sizeof(TrainState))) ||
        (rc = c->packed_fwd.ensure(kFwdSize * 2)) || (rc = c->packed_bwd.ensure(kBwdSize * 2)) ||
        (rc = c->bias.ensure(kBiasSteps * sizeof(float2)))) {
        delete c;
        return rc;
    }
    // zero fragments that no weight maps to (padded rows/columns)
    if (hipMemset(c->packed_fwd.ptr, 0, kFwdSize * 2) != hipSuccess ||
        hipMemset(c->packed_bwd.ptr, 0, kBwdSize * 2) != hipSuccess) {
        delete c;
        return set_error(CUPBR_ERR_HIP, "hipMemset failed");
    }
    // Adam's bias corrections, one pair per step number (every cache has the same betas)
    static const std::vector<float2> bias = [](float b1, float b2) {
        std::vector<float2> t(kBiasSteps);
        for (uint32_t k = 0; k < kBiasSteps; ++k)
            t[k] = make_float2(1.0f - std::pow(b1, (float)k), 1.0f - std::pow(b2, (float)k));
        return t;
    }(c->beta1, c->beta2);
    if (hipMemcpy(c->bias.ptr, bias.data(), kBiasSteps * sizeof(float2), hipMemcpyHostToDevice) != hipSuccess) {
        delete c;
        return set_error(CUPBR_ERR_HIP, "hipMemcpy failed");
    }
    if ((rc = nrc_init_weights(c, seed))) {
        delete c;
        return rc;
    }
    CUPBR_HIP_CHECK(hipDeviceSynchronize());
    *out = c;
    return CUPBR_OK;
}

int nrc_infer(cupbr_nrc* c, const float* rec, uint32_t n, const uint32_t* n_dev, uint32_t stride, float* out,
              bool accumulate, hipStream_t stream, const uint32_t* begin_dev, NrcParts parts) {
    if (n == 0) return CUPBR_OK;
    const uint32_t pairs = (n + 31) / 32;  // a wave takes two 16-query tiles at a time
    uint32_t blocks = std::max<uint32_t>(1, std::min<uint32_t>((pairs + 3) / 4, (uint32_t)device_cu_count() * 2));
    if (parts.size != 0) blocks = (blocks + 7) / 8 * 8;
    if (accumulate)
        hipLaunchKernelGGL(k_nrc_infer<true>, dim3(blocks), dim3(kNrcBlock), 0, stream, c->packed_fwd.as<bf16x8>(),
                           c->box, rec, n, n_dev, stride, out, begin_dev, parts);
    else
        hipLaunchKernelGGL(k_nrc_infer<false>, dim3(blocks), dim3(kNrcBlock), 0, stream, c->packed_fwd.as<bf16x8>(),
                           c->box, rec, n, n_dev, stride, out, begin_dev, parts);
    CUPBR_HIP_CHECK(hipGetLastError());
    return CUPBR_OK;
}

int nrc_train(cupbr_nrc* c, const float* rows, uint32_t n_rows, uint32_t batch, uint32_t steps, float lr,
              float* loss_dev, hipStream_t stream, const uint32_t* n_rows_dev) {
    if (n_rows == 0 || steps == 0) return CUPBR_OK;
    // a block per 64 rows, in groups of 8 slices, at most about one per CU (its 149 KB of LDS allow no second one)
    const uint32_t n_slices = batch / kSlice, groups = (n_slices + 7) / 8;
    const uint32_t blocks = 64 * std::min<uint32_t>(groups, std::max(1u, (uint32_t)device_cu_count() / 64));
    int rc;
    if ((rc = c->acts.ensure((size_t)n_slices * kOperands * kSliceOperand * 16)) || (rc = c->losses.ensure((size_t)blocks * 4)) ||
        (rc = c->sums.ensure((size_t)kWeightTiles * (batch / kSlice) * 1024)))
        return rc;
    const uint32_t sum_blocks = groups * 8 * (kWeightTiles / 4);
    float *m = c->moments.as<float>(), *v = m + kNrcParams;
    TrainState* state = reinterpret_cast<TrainState*>(v + kNrcParams);
    for (uint32_t s = 0; s < steps; ++s) {
        hipLaunchKernelGGL(k_nrc_train, dim3(blocks), dim3(kNrcBlock), 0, stream, c->packed_fwd.as<bf16x8>(),
                           c->packed_bwd.as<bf16x8>(), c->box, rows, n_rows, n_rows_dev, batch, state, s,
                           c->acts.as<bf16x8>(), c->losses.as<float>());
        CUPBR_HIP_CHECK(hipGetLastError());
        hipLaunchKernelGGL(k_nrc_weight_sums, dim3(sum_blocks), dim3(kNrcBlock), 0, stream, c->acts.as<bf16x8>(), n_slices,
                           c->sums.as<f32x4>(), n_rows, n_rows_dev);
        CUPBR_HIP_CHECK(hipGetLastError());
        hipLaunchKernelGGL(k_nrc_adam, dim3(kWeightTiles + 1), dim3(kNrcBlock), 0, stream, c->sums.as<f32x4>(), n_slices,
                           c->losses.as<float>(), blocks, 1.0f / (float)batch, c->w.as<float>(), m, v, lr, c->beta1, c->beta2, c->eps, c->bias.as<float2>(), n_rows, n_rows_dev,
                           state, s + 1 == steps ? steps : 0u, loss_dev ? loss_dev + s : nullptr,
                           c->packed_fwd.as<__bf16>(), c->packed_bwd.as<__bf16>());
        CUPBR_HIP_CHECK(hipGetLastError());
    }
    return CUPBR_OK;
}

int nrc_mfma_product(const float* a, const float* b, float* d) {
    DevBuf da, db, dd;
    int rc;
    if ((rc = da.ensure(16 * 32 * 4)) || (rc = db.ensure(32 * 16 * 4)) || (rc = dd.ensure(16 * 16 * 4))) return rc;
    CUPBR_HIP_CHECK(hipMemcpy(da.ptr, a, 16 * 32 * 4, hipMemcpyHostToDevice));
    CUPBR_HIP_CHECK(hipMemcpy(db.ptr, b, 32 * 16 * 4, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(k_nrc_mfma_product, dim3(1), dim3(64), 0, nullptr, da.as<float>(), db.as<float>(), dd.as<float>());
    CUPBR_HIP_CHECK(hipGetLastError());
    CUPBR_HIP_CHECK(hipMemcpy(d, dd.ptr, 16 * 16 * 4, hipMemcpyDeviceToHost));
    return CUPBR_OK;
}

}  // namespace cupbr
