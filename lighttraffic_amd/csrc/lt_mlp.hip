// lt_mlp.hip — training and inference kernels of the learned partition scorer.
//
// Layers (row-major, input-major weights: y[j] = sum_k x[k] W[k][j] + b[j]):
//   X[M x 16] -> A1 = relu(X W1 + b1) [M x 256] -> A2 = relu(A1 W2 + b2)
//   -> Y = A2 W3 + b3 [M x 2],   M = (decisions in a batch) x P partitions.
// Weights are kept as FP32 masters for Adam and used as their BF16 rounding
// (round to nearest even) in every product; products accumulate in FP32.
// Losses per decision: softmax cross-entropy of output 0 over the partitions
// holding walkers against the partition the plain scheduler picked next, and
// mean squared error of output 1 against the partition's future traffic share.
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <memory>
#include <mutex>
#include <random>
#include <vector>

#include "lt_internal.h"
#include "lt_mlp.h"

#define LT_NA_TRY(expr)             \
    do {                            \
        lt_status _s = (expr);      \
        if (_s != LT_OK) return _s; \
    } while (0)

#define MLP_HIP(call)                                                                                  \
    do {                                                                                               \
        hipError_t _e = (call);                                                                        \
        if (_e != hipSuccess) {                                                                        \
            lt::set_error("%s:%d %s: %s", __FILE__, __LINE__, #call, hipGetErrorString(_e));            \
            return LT_E_HIP;                                                                           \
        }                                                                                              \
    } while (0)

namespace lt {

// ---- parameter layout ------------------------------------------------------
constexpr size_t kOffW1 = 0;
constexpr size_t kOffB1 = kOffW1 + (size_t)kFeat * kHidden;
constexpr size_t kOffW2 = kOffB1 + kHidden;
constexpr size_t kOffB2 = kOffW2 + (size_t)kHidden * kHidden;
constexpr size_t kOffW3 = kOffB2 + kHidden;
constexpr size_t kOffB3 = kOffW3 + (size_t)kHidden * kOut;
constexpr size_t kParams = kOffB3 + kOut;

__host__ __device__ inline uint16_t f32_to_bf16(float x) {
    uint32_t u;
    memcpy(&u, &x, 4);
    if ((u & 0x7F800000u) == 0x7F800000u && (u & 0x007FFFFFu)) return (uint16_t)((u >> 16) | 0x40u);  // NaN stays NaN
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__device__ __forceinline__ float bf16_to_f32(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// ---- features ----------------------------------------------------------------
// Feature j of partition q:
//  0 log1p(c)/log1p(W)   1 c/max c   2 log1p(c/mean c)   3 resident
//  4 chosen now          5..11 loaded k decisions ago (k = 0..6)
//  12 a/(a+P), a = HBM walks since q's last one (recency: Belady's victim is
//     the partition needed farthest ahead, and on walk schedules that is
//     mostly the one walked longest ago)
//  13 vertex share * P   14 edge share * P   15 queued walkers / W
constexpr int kRecentFeat = 7;  // recent loads that become features (the state holds kRecent)

__device__ __forceinline__ float age_feature(uint32_t a, uint32_t P) { return (float)a / ((float)a + (float)P); }

// Copy of the first two layers' weights, output-major: Wi[j * kFeat + k] =
// W1[k][j] and Wi[kWiW2 + j * kHidden + k] = W2[k][j], so that the
// weights of output j come in 16-byte loads.
constexpr size_t kWiW2 = (size_t)kHidden * kFeat;
constexpr size_t kWiSize = kWiW2 + (size_t)kHidden * kHidden;

// ---- training ------------------------------------------------------------------
// One step over M = decisions * P rows in four launches:
//   train_forward_kernel   features and the three layers, 32 rows per workgroup
//   loss_kernel            losses and dY, one workgroup per decision
//   train_backward_kernel  two kinds of workgroups: tiles of 32 rows, dA2 and
//                          dA1 with their part of every gradient but W2's; and a
//                          quarter of W2's gradient over a slice of the rows
//   train_update_kernel    the gradient (partial sums added in a fixed order),
//                          and Adam
// Products run on the matrix cores in FP32 (v_mfma_f32_32x32x2_f32: FP32
// inputs and accumulation, as on the vector units).  Bound: at 32 decisions of
// 291 partitions the 3.8 GFLOP take 24 us at the FP32 matrix rate; these launches
// take 33, 11, 53 and 13, and the sixteen of 64 x 64 LDS-tiled vector GEMMs and
// their split-K sums took 460.  The batch is read in place from pinned memory
// (121 KB; a copy to the device first measured the same in all, ten separate
// copies 150 us more).
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kTileRows = 32;
constexpr int kLdH = kHidden + 4;  // LDS row of 256 columns: 16-byte aligned, rows 4 banks apart
constexpr uint32_t kSliceMost = 64;   // slices of the rows in W2's gradient: 4 x 64 workgroups fill the chip
constexpr uint32_t kGroupMost = 512;  // workgroups of the other kind, two per CU
constexpr int kSmallParams = (int)kParams - kHidden * kHidden;  // all but W2

// The small gradients' order in a partial row: W1, b1, b2, W3, b3.
constexpr int kSmB1 = kFeat * kHidden, kSmB2 = kSmB1 + kHidden, kSmW3 = kSmB2 + kHidden, kSmB3 = kSmW3 + kHidden * kOut;

// One batch of decisions in mapped host memory (stage_batch).
struct Batch {
    const uint32_t *counts, *age;  // [n][P]
    const float *keep;             // [n][P]
    const float *scale;            // [n][3]: walkers, largest count, sum of the counts
    const int32_t *recent;         // [n][kRecent]
    const int32_t *cur, *next;     // [n]
    const float *wa, *wb;          // [n]
    const uint8_t *resident;       // [n][P]
};

// Features of partition q; head gives the decision's scalars.
__device__ __forceinline__ void features(float *x, uint32_t P, uint32_t q, uint32_t count, bool res, uint32_t age,
                                         float w_total, float max_count, float sum, int32_t cur, const int32_t *recent,
                                         float vsh, float esh) {
    const float W = fmaxf(w_total, 1.f);
    const float cmax = fmaxf(max_count, 1.f);
    const float mean = fmaxf(sum / (float)P, 1.f);
    const float v = (float)count;
    x[0] = log1pf(v) / log1pf(W);
    x[1] = v / cmax;
    x[2] = log1pf(v / mean);
    x[3] = res ? 1.f : 0.f;
    x[4] = cur == (int32_t)q ? 1.f : 0.f;
#pragma unroll
    for (int k = 0; k < kRecentFeat; k++) x[5 + k] = recent[k] == (int32_t)q ? 1.f : 0.f;
    x[12] = age_feature(age, P);
    x[13] = vsh;
    x[14] = esh;
    x[15] = sum / W;
}

__device__ __forceinline__ void unpack8(const uint4 &w, float *f) {
    const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        f[2 * i] = __uint_as_float(u[i] << 16);
        f[2 * i + 1] = __uint_as_float(u[i] & 0xFFFF0000u);
    }
}

// acc[t] += A[32 x 256] * B for the wave's two 32-column tiles: A is an LDS
// tile of kLdH-float rows, B[k][n] = bt[n * 256 + k] (BF16).  In a step of 64 k
// the lanes of a wave's lower half hold k = 64 s .. +31 and those of its upper
// half the next 32, for A and B alike: a lane reads 64 bytes of one weight row
// at a time, and the next step's weights arrive while this one's 64 products
// run (1.7 us).  The first step's weights the caller loads ahead.
struct WeightStep {
    uint4 w0[4], w1[4];
};
__device__ __forceinline__ WeightStep first_weights(const uint16_t *bt, int n0) {
    const int lane = threadIdx.x & 63, i = lane & 31, h = lane >> 5;
    WeightStep w;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        w.w0[c] = ((const uint4 *)(bt + (size_t)(n0 + i) * kHidden + 32 * h))[c];
        w.w1[c] = ((const uint4 *)(bt + (size_t)(n0 + 32 + i) * kHidden + 32 * h))[c];
    }
    return w;
}
__device__ __forceinline__ void mfma_rows(const float *sA, const uint16_t *bt, int n0, const WeightStep &first,
                                          f32x16 (&acc)[2]) {
    const int lane = threadIdx.x & 63, i = lane & 31, h = lane >> 5;
    const uint4 *b0 = (const uint4 *)(bt + (size_t)(n0 + i) * kHidden + 32 * h);
    const uint4 *b1 = (const uint4 *)(bt + (size_t)(n0 + 32 + i) * kHidden + 32 * h);
    const float *a = sA + i * kLdH + 32 * h;
    uint4 w0[4], w1[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
        w0[c] = first.w0[c];
        w1[c] = first.w1[c];
    }
#pragma unroll
    for (int s = 0; s < kHidden / 64; s++) {
        uint4 v0[4], v1[4];
        if (s + 1 < kHidden / 64) {
#pragma unroll
            for (int c = 0; c < 4; c++) {
                v0[c] = b0[8 * (s + 1) + c];
                v1[c] = b1[8 * (s + 1) + c];
            }
        }
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const float4 lo = *(const float4 *)(a + 64 * s + 8 * c), hi = *(const float4 *)(a + 64 * s + 8 * c + 4);
            const float av[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
            float f0[8], f1[8];
            unpack8(w0[c], f0);
            unpack8(w1[c], f1);
#pragma unroll
            for (int j = 0; j < 8; j++) {
                acc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[j], f0[j], acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[j], f1[j], acc[1], 0, 0, 0);
            }
        }
        if (s + 1 < kHidden / 64) {
#pragma unroll
            for (int c = 0; c < 4; c++) {
                w0[c] = v0[c];
                w1[c] = v1[c];
            }
        }
    }
}

// Row of element r of a 32 x 32 result tile (column = lane % 32).
__device__ __forceinline__ int tile_row(int r) { return 8 * (r >> 2) + 4 * ((int)(threadIdx.x & 63) >> 5) + (r & 3); }

__global__ __launch_bounds__(256) void train_forward_kernel(uint32_t P, uint32_t M, Batch d, const float *vsh,
                                                            const float *esh, const uint16_t *Wb, const uint16_t *Wi,
                                                            uint32_t *counts, float *X, float *A1, float *A2,
                                                            float *Y) {
    __shared__ __align__(16) float s_x[kTileRows][kFeat + 1];
    __shared__ __align__(16) float s_a[kTileRows * kLdH];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i = lane & 31, h = lane >> 5;
    const int n0 = wave * 64;
    // weights do not wait for the features
    const uint4 w1[2] = {*(const uint4 *)(Wi + (size_t)(n0 + i) * kFeat + 8 * h),
                         *(const uint4 *)(Wi + (size_t)(n0 + 32 + i) * kFeat + 8 * h)};
    const WeightStep w2 = first_weights(Wi + kWiW2, n0);
    const float bias1[2] = {bf16_to_f32(Wb[kOffB1 + n0 + i]), bf16_to_f32(Wb[kOffB1 + n0 + 32 + i])};
    const float bias2[2] = {bf16_to_f32(Wb[kOffB2 + n0 + i]), bf16_to_f32(Wb[kOffB2 + n0 + 32 + i])};
    const uint32_t r0 = blockIdx.x * kTileRows;
    if (tid < kTileRows) {
        const uint32_t r = r0 + tid;
        float x[kFeat];
#pragma unroll
        for (int k = 0; k < kFeat; k++) x[k] = 0.f;
        if (r < M) {
            const uint32_t b = r / P, q = r - b * P;
            const uint32_t count = d.counts[r];
            counts[r] = count;
            features(x, P, q, count, d.resident[r], d.age[r], d.scale[3 * b], d.scale[3 * b + 1],
                     d.scale[3 * b + 2], d.cur[b], d.recent + b * kRecent, vsh[q], esh[q]);
        }
#pragma unroll
        for (int k = 0; k < kFeat; k++) s_x[tid][k] = x[k];
    }
    __syncthreads();
    for (int t = tid; t < kTileRows * kFeat; t += 256)
        if (r0 + t / kFeat < M) X[(size_t)r0 * kFeat + t] = s_x[t / kFeat][t % kFeat];
    f32x16 acc[2] = {};
#pragma unroll
    for (int t = 0; t < 2; t++) {
        float f[8];
        unpack8(w1[t], f);
#pragma unroll
        for (int j = 0; j < 8; j++)
            acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(s_x[i][8 * h + j], f[j], acc[t], 0, 0, 0);
    }
    const auto layer_out = [&](const float (&bias)[2], float *A) {
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int n = n0 + 32 * t + i;
            const float bn = bias[t];
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int m = tile_row(r);
                const float v = fmaxf(acc[t][r] + bn, 0.f);
                s_a[m * kLdH + n] = v;
                if (r0 + m < M) A[(size_t)(r0 + m) * kHidden + n] = v;
            }
        }
    };
    layer_out(bias1, A1);
    __syncthreads();
    acc[0] = acc[1] = f32x16{};
    mfma_rows(s_a, Wi + kWiW2, n0, w2, acc);
    __syncthreads();
    layer_out(bias2, A2);
    __syncthreads();
    const int row = tid >> 3, part = tid & 7;  // eight threads per row, 4 of every 32 columns each
    float y0 = 0.f, y1 = 0.f;
#pragma unroll
    for (int s = 0; s < kHidden / 32; s++) {
        const int k = 32 * s + 4 * part;
        const float4 v = *(const float4 *)(s_a + row * kLdH + k);
        float w[8];
        unpack8(*(const uint4 *)(Wb + kOffW3 + k * kOut), w);
        y0 = fmaf(v.x, w[0], y0);
        y1 = fmaf(v.x, w[1], y1);
        y0 = fmaf(v.y, w[2], y0);
        y1 = fmaf(v.y, w[3], y1);
        y0 = fmaf(v.z, w[4], y0);
        y1 = fmaf(v.z, w[5], y1);
        y0 = fmaf(v.w, w[6], y0);
        y1 = fmaf(v.w, w[7], y1);
    }
#pragma unroll
    for (int off = 1; off < 8; off <<= 1) {
        y0 += __shfl_xor(y0, off, 64);
        y1 += __shfl_xor(y1, off, 64);
    }
    if (part == 0 && r0 + row < M)
        ((float2 *)Y)[r0 + row] = make_float2(y0 + bf16_to_f32(Wb[kOffB3]), y1 + bf16_to_f32(Wb[kOffB3 + 1]));
}

// dA2[m][n] before the ReLU mask.
__device__ __forceinline__ float back3(float dy0, float dy1, float w0, float w1) { return fmaf(dy1, w1, dy0 * w0); }

__global__ __launch_bounds__(256, 2) void train_backward_kernel(uint32_t M, uint32_t groups, uint32_t slices,
                                                             const float *X, const float *A1, const float *A2,
                                                             const float *dY, const uint16_t *Wb, float *small,
                                                             float *w2) {
    __shared__ __align__(16) float s_d2[kTileRows * kLdH];
    __shared__ __align__(16) float s_d1[kTileRows * kLdH];
    __shared__ __align__(16) float s_x[kTileRows][kFeat];
    __shared__ float s_dy[kTileRows][kOut];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i = lane & 31, h = lane >> 5;
    const uint32_t tiles = (M + kTileRows - 1) / kTileRows;
    if (blockIdx.x < groups) {
        float g[kFeat] = {}, b1 = 0.f, b2 = 0.f, b3 = 0.f, g0 = 0.f, g1 = 0.f;
        const float w30 = bf16_to_f32(Wb[kOffW3 + tid * kOut]), w31 = bf16_to_f32(Wb[kOffW3 + tid * kOut + 1]);
        const int n0 = wave * 64;
        const WeightStep w2t = first_weights(Wb + kOffW2, n0);
        for (uint32_t tile = blockIdx.x; tile < tiles; tile += groups) {
            const uint32_t r0 = tile * kTileRows;
            const int rows = (int)min((uint32_t)kTileRows, M - r0);
            // everything the tile reads is on its way before any of it is waited for
            float a2[kTileRows];
#pragma unroll
            for (int m = 0; m < kTileRows; m++) a2[m] = m < rows ? A2[(size_t)(r0 + m) * kHidden + tid] : 0.f;
            uint32_t on = 0;  // ReLU masks of this lane's 32 elements of dA1
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int m = tile_row(r);
                    if (m < rows && A1[(size_t)(r0 + m) * kHidden + n0 + 32 * t + i] > 0.f) on |= 1u << (16 * t + r);
                }
            for (int t = tid; t < kTileRows * kFeat; t += 256)
                s_x[t / kFeat][t % kFeat] = t / kFeat < rows ? X[(size_t)r0 * kFeat + t] : 0.f;
            if (tid < kTileRows * kOut)
                s_dy[tid / kOut][tid % kOut] = tid / kOut < rows ? dY[(size_t)r0 * kOut + tid] : 0.f;
            __syncthreads();
            // thread = column: dA2, and the sums over its rows that need no product
#pragma unroll
            for (int m = 0; m < kTileRows; m++) {
                const float y0 = s_dy[m][0], y1 = s_dy[m][1];
                const float v = a2[m] > 0.f ? back3(y0, y1, w30, w31) : 0.f;
                s_d2[m * kLdH + tid] = v;
                b2 += v;
                g0 = fmaf(a2[m], y0, g0);
                g1 = fmaf(a2[m], y1, g1);
            }
            if (tid < kOut)
                for (int m = 0; m < kTileRows; m++) b3 += s_dy[m][tid];
            __syncthreads();
            f32x16 acc[2] = {};
            mfma_rows(s_d2, Wb + kOffW2, n0, w2t, acc);  // dA1[m][j] = sum_n dA2[m][n] W2[j][n]
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 16; r++)
                    s_d1[tile_row(r) * kLdH + n0 + 32 * t + i] = (on >> (16 * t + r)) & 1u ? acc[t][r] : 0.f;
            __syncthreads();
#pragma unroll 8
            for (int m = 0; m < kTileRows; m++) {
                const float v = s_d1[m * kLdH + tid];
                b1 += v;
#pragma unroll
                for (int f = 0; f < kFeat; f++) g[f] = fmaf(s_x[m][f], v, g[f]);
            }
            __syncthreads();
        }
        float *out = small + (size_t)blockIdx.x * kSmallParams;
#pragma unroll
        for (int f = 0; f < kFeat; f++) out[f * kHidden + tid] = g[f];
        out[kSmB1 + tid] = b1;
        out[kSmB2 + tid] = b2;
        out[kSmW3 + tid * kOut] = g0;
        out[kSmW3 + tid * kOut + 1] = g1;
        if (tid < kOut) out[kSmB3 + tid] = b3;
        return;
    }
    // W2's gradient: slice z of the row tiles, 128 x 128 quarter (k0, n0); each
    // wave 64 x 64 of it.  The next tile's rows are loaded while this one's
    // products run.
    const uint32_t z = (blockIdx.x - groups) >> 2, quarter = (blockIdx.x - groups) & 3;
    const int k0 = (int)(quarter >> 1) * 128, n0 = (int)(quarter & 1) * 128;
    const uint32_t t0 = (uint32_t)((uint64_t)tiles * z / slices), t1 = (uint32_t)((uint64_t)tiles * (z + 1) / slices);
    constexpr int kLdT = 128, kHalf = kTileRows / 2;  // LDS row of a staged tile; its rows per thread
    float *s_a = s_d2, *s_b = s_d1;
    const int wk = (wave >> 1) * 64, wn = (wave & 1) * 64;
    const int c = tid & 127, half = tid >> 7;
    const float w30 = bf16_to_f32(Wb[kOffW3 + (n0 + c) * kOut]), w31 = bf16_to_f32(Wb[kOffW3 + (n0 + c) * kOut + 1]);
    float a[kHalf], b[kHalf];
    float2 dy[kHalf];
    const auto load = [&](uint32_t t) {
        const uint32_t r0 = t * kTileRows;
#pragma unroll
        for (int m = 0; m < kHalf; m++) {
            const uint32_t r = r0 + 2 * m + half;
            const bool in = r < M;
            a[m] = in ? A1[(size_t)r * kHidden + k0 + c] : 0.f;
            b[m] = in ? A2[(size_t)r * kHidden + n0 + c] : 0.f;
            dy[m] = in ? ((const float2 *)dY)[r] : make_float2(0.f, 0.f);
        }
    };
    f32x16 acc[2][2] = {};
    load(t0);
    for (uint32_t t = t0; t < t1; t++) {
        __syncthreads();
#pragma unroll
        for (int m = 0; m < kHalf; m++) {
            s_a[(2 * m + half) * kLdT + c] = a[m];
            s_b[(2 * m + half) * kLdT + c] = b[m] > 0.f ? back3(dy[m].x, dy[m].y, w30, w31) : 0.f;
        }
        __syncthreads();
        if (t + 1 < t1) load(t + 1);
#pragma unroll
        for (int s = 0; s < kHalf; s++) {
            const float *ra = s_a + (2 * s + h) * kLdT + wk + i, *rb = s_b + (2 * s + h) * kLdT + wn + i;
            const float a0 = ra[0], a1 = ra[32], b0 = rb[0], b1 = rb[32];
            acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, b0, acc[0][0], 0, 0, 0);
            acc[0][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, b1, acc[0][1], 0, 0, 0);
            acc[1][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, b0, acc[1][0], 0, 0, 0);
            acc[1][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, b1, acc[1][1], 0, 0, 0);
        }
    }
    float *out = w2 + (size_t)z * kHidden * kHidden;
#pragma unroll
    for (int ta = 0; ta < 2; ta++)
#pragma unroll
        for (int tb = 0; tb < 2; tb++)
#pragma unroll
            for (int r = 0; r < 16; r++)
                out[(size_t)(k0 + wk + 32 * ta + tile_row(r)) * kHidden + n0 + wn + 32 * tb + i] = acc[ta][tb][r];
}

// Gradient of 32 parameters per workgroup: 8 threads share a parameter's
// partial sums, added in a fixed order.  With update, Adam on them (their
// BF16 forms included); host: the gradient goes there too.  The first workgroup
// adds up the decisions' losses.
__global__ __launch_bounds__(256) void train_update_kernel(uint32_t groups, uint32_t slices, const float *small,
                                                           const float *w2, float *host, float *W,
                                                           uint16_t *Wb, uint16_t *Wi, float *Mo, float *Vo, int update,
                                                           float lr, float b1t, float b2t, uint32_t n,
                                                           const float *losses, float *loss) {
    __shared__ float s_p[8][32];
    const int c = threadIdx.x & 31, g = threadIdx.x >> 5;
    const uint32_t p = blockIdx.x * 32 + c;
    float sum = 0.f;
    if (p < kParams) {
        const bool is_w2 = p >= kOffW2 && p < kOffB2;
        // partial rows hold the parameters without W2 in the same order
        const float *q = is_w2 ? w2 + (p - kOffW2) : small + (p < kOffW2 ? p : p - kHidden * kHidden);
        const size_t ld = is_w2 ? (size_t)kHidden * kHidden : (size_t)kSmallParams;
        const uint32_t parts = is_w2 ? slices : groups;
        uint32_t k = g;
        for (; k + 24 < parts; k += 32) {  // four loads in flight
            const float x0 = q[k * ld], x1 = q[(k + 8) * ld], x2 = q[(k + 16) * ld], x3 = q[(k + 24) * ld];
            sum += (x0 + x1) + (x2 + x3);
        }
        for (; k < parts; k += 8) sum += q[k * ld];
    }
    s_p[g][c] = sum;
    __syncthreads();
    if (g == 0 && p < kParams) {
        float s = 0.f;
#pragma unroll
        for (int k = 0; k < 8; k++) s += s_p[k][c];
        if (host) host[p] = s;
        if (update) {
            const float m = 0.9f * Mo[p] + 0.1f * s;
            const float v = 0.999f * Vo[p] + 0.001f * s * s;
            Mo[p] = m;
            Vo[p] = v;
            const float w = W[p] - lr * (m / (1.f - b1t)) / (sqrtf(v / (1.f - b2t)) + 1e-8f);
            W[p] = w;
            const uint16_t r = f32_to_bf16(w);
            Wb[p] = r;
            if (p < kOffB1) Wi[(p % kHidden) * kFeat + p / kHidden] = r;
            else if (p >= kOffW2 && p < kOffB2)
                Wi[kWiW2 + ((p - kOffW2) % kHidden) * kHidden + (p - kOffW2) / kHidden] = r;
        }
    }
    if (blockIdx.x == 0 && threadIdx.x < 64) {
        float l[2] = {0.f, 0.f};
        for (uint32_t b = threadIdx.x; b < n; b += 64) {
            l[0] += losses[2 * b];
            l[1] += losses[2 * b + 1];
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            l[0] += __shfl_xor(l[0], off, 64);
            l[1] += __shfl_xor(l[1], off, 64);
        }
        if (threadIdx.x < 2) loss[threadIdx.x] = l[threadIdx.x];
    }
}

// ---- losses -----------------------------------------------------------------
// One workgroup per decision; writes dY and the decision's weighted losses.
__global__ __launch_bounds__(256) void loss_kernel(uint32_t P, uint32_t B, const float *Y, const uint32_t *counts,
                                                   const int32_t *next_label, const float *keep_label,
                                                   const float *wa, const float *wb, float *dY, float *losses) {
    const uint32_t b = blockIdx.x;
    const float *y = Y + (size_t)b * P * kOut;
    float *dy = dY + (size_t)b * P * kOut;
    const uint32_t *c = counts + (size_t)b * P;
    const int32_t lab = next_label[b];
    const float a_w = lab >= 0 ? wa[b] : 0.f, b_w = wb[b];
    __shared__ float s_red[3][4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // softmax over candidates (walkers queued, or the label itself)
    float mx = -INFINITY;
    for (uint32_t q = threadIdx.x; q < P; q += blockDim.x)
        if (c[q] > 0 || (int32_t)q == lab) mx = fmaxf(mx, y[q * kOut]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
    if (lane == 0) s_red[0][wave] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(s_red[0][0], s_red[0][1]), fmaxf(s_red[0][2], s_red[0][3]));
    float se = 0.f;
    for (uint32_t q = threadIdx.x; q < P; q += blockDim.x)
        if (c[q] > 0 || (int32_t)q == lab) se += expf(y[q * kOut] - mx);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) se += __shfl_xor(se, off, 64);
    if (lane == 0) s_red[1][wave] = se;
    __syncthreads();
    se = (s_red[1][0] + s_red[1][1]) + (s_red[1][2] + s_red[1][3]);
    float lb = 0.f;
    const float inv_b = 1.f / (float)B;
    for (uint32_t q = threadIdx.x; q < P; q += blockDim.x) {
        const bool cand = c[q] > 0 || (int32_t)q == lab;
        float g0 = 0.f;
        if (cand && a_w > 0.f && se > 0.f) {
            const float p = expf(y[q * kOut] - mx) / se;
            g0 = a_w * (p - ((int32_t)q == lab ? 1.f : 0.f)) * inv_b;
        }
        const float d = y[q * kOut + 1] - keep_label[(size_t)b * P + q];
        lb += b_w * d * d;
        dy[q * kOut] = g0;
        dy[q * kOut + 1] = b_w * 2.f * d * inv_b / (float)P;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) lb += __shfl_xor(lb, off, 64);
    if (lane == 0) s_red[2][wave] = lb;
    __syncthreads();
    lb = (s_red[2][0] + s_red[2][1]) + (s_red[2][2] + s_red[2][3]);
    if (threadIdx.x == 0) {
        losses[2 * b] = a_w > 0.f && se > 0.f ? a_w * (logf(se) + mx - y[lab * kOut]) * inv_b : 0.f;
        losses[2 * b + 1] = lb * inv_b / (float)P;
    }
}

__global__ void round_kernel(size_t n, const float *W, uint16_t *Wb) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) Wb[i] = f32_to_bf16(W[i]);
}

// ---- fused inference: one decision, R partitions per workgroup --------------
__global__ void transpose_infer_weights_kernel(const uint16_t *Wb, uint16_t *Wi) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < kWiW2) {
        const size_t j = i / kFeat, k = i % kFeat;
        Wi[i] = Wb[kOffW1 + k * kHidden + j];
    } else if (i < kWiSize) {
        const size_t t = i - kWiW2, j = t / kHidden, k = t % kHidden;
        Wi[i] = Wb[kOffW2 + k * kHidden + j];
    }
}

// The decision state infer_kernel reads, packed in one buffer (host memory
// mapped for the device, or device memory):
//   i32 recent[8] | i32 cur | f32 w_total | f32 max count | f32 count sum |
//   pad to kStateHead | u32 counts[P] | u32 age[P] | u8 resident[P]
// The host supplies the max and the sum of the counts, so a workgroup reads
// only the header and its own rows: the launch reads O(P) bytes of the state,
// and LDS use does not grow with P.
constexpr size_t kStateHead = 64;
constexpr int kHeadCur = kRecent, kHeadW = kRecent + 1, kHeadMax = kRecent + 2, kHeadSum = kRecent + 3;
static_assert(4 * (kHeadSum + 1) <= (int)kStateHead, "state header");
__host__ __device__ constexpr size_t state_bytes(uint32_t P) { return kStateHead + 9 * (size_t)P; }

// Header of one decision's packed state.
static void pack_state_head(int32_t *head, const uint32_t *counts, uint32_t P, const int32_t *recent, int32_t cur,
                            float w_total) {
    uint32_t mx = 0;
    double sum = 0.0;
    for (uint32_t q = 0; q < P; q++) {
        mx = std::max(mx, counts[q]);
        sum += counts[q];
    }
    memset(head, 0, kStateHead);
    for (int k = 0; k < kRecent; k++) head[k] = recent[k];
    head[kHeadCur] = cur;
    const float f[3] = {w_total, (float)mx, (float)sum};
    memcpy(&head[kHeadW], f, sizeof(f));
}

// Each workgroup builds the features of R partitions (rows) and runs the
// three layers on them.  Each output neuron accumulates its inputs in
// increasing order in FP32, whatever R.  A decision waits for this kernel: with
// 8 rows 291 partitions keep 37 of 256 CUs busy for 17 us, with 2 rows 146 for
// 10.6.  Above kFewRows partitions there are workgroups enough, and 8 rows share
// the weights: calls with 2 rows and with 8 take 22.4 and 28.0 us for 512 partitions, 27.1
// and 28.8 for 1,024, 30.7 and 29.0 for 1,100, 58 and 36 for 4,096, 214 and 112 for 20,000.
template <int R>
__global__ __launch_bounds__(256) void infer_kernel(uint32_t P, const uint8_t *state, const float *vsh,
                                                    const float *esh, const uint16_t *Wb, const uint16_t *Wi,
                                                    float *Y) {
    __shared__ float s_x[R][kFeat];
    __shared__ float s_h1[R][kHidden];
    __shared__ float s_h2[R][kHidden];
    const int j = threadIdx.x;
    const int32_t *head = (const int32_t *)state;
    const uint32_t *counts = (const uint32_t *)(state + kStateHead);
    const uint32_t *age = counts + P;
    const uint8_t *res = state + kStateHead + 8 * (size_t)P;
    const uint32_t r0 = blockIdx.x * R;
    if (j < R) {
        const uint32_t q = r0 + j;
        float *x = s_x[j];
        if (q < P) {
            features(x, P, q, counts[q], res[q], age[q], __int_as_float(head[kHeadW]), __int_as_float(head[kHeadMax]),
                     __int_as_float(head[kHeadSum]), head[kHeadCur], head, vsh[q], esh[q]);
        } else {
            for (int k = 0; k < kFeat; k++) x[k] = 0.f;
        }
    }
    __syncthreads();
    const uint16_t *B1 = Wb + kOffB1, *B2 = Wb + kOffB2, *W3 = Wb + kOffW3, *B3 = Wb + kOffB3;
    float a[R];
#pragma unroll
    for (int r = 0; r < R; r++) a[r] = 0.f;
    {
        const uint4 *w1 = (const uint4 *)(Wi + (size_t)j * kFeat);
        uint4 wv[kFeat / 8];
#pragma unroll
        for (int c = 0; c < kFeat / 8; c++) wv[c] = w1[c];
#pragma unroll
        for (int k = 0; k < kFeat; k++) {
            const uint32_t word = (&wv[k / 8].x)[(k % 8) / 2];
            const float w = __uint_as_float((k & 1) ? (word & 0xFFFF0000u) : (word << 16));
#pragma unroll
            for (int r = 0; r < R; r++) a[r] = fmaf(s_x[r][k], w, a[r]);
        }
    }
#pragma unroll
    for (int r = 0; r < R; r++) s_h1[r][j] = fmaxf(a[r] + bf16_to_f32(B1[j]), 0.f);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; r++) a[r] = 0.f;
    const uint4 *w2 = (const uint4 *)(Wi + kWiW2 + (size_t)j * kHidden);
    for (int k0 = 0; k0 < kHidden; k0 += 64) {
        uint4 wv[8];
#pragma unroll
        for (int c = 0; c < 8; c++) wv[c] = w2[k0 / 8 + c];
#pragma unroll
        for (int kk = 0; kk < 64; kk++) {
            const uint32_t word = (&wv[kk / 8].x)[(kk % 8) / 2];
            const float w = __uint_as_float((kk & 1) ? (word & 0xFFFF0000u) : (word << 16));
#pragma unroll
            for (int r = 0; r < R; r++) a[r] = fmaf(s_h1[r][k0 + kk], w, a[r]);
        }
    }
#pragma unroll
    for (int r = 0; r < R; r++) s_h2[r][j] = fmaxf(a[r] + bf16_to_f32(B2[j]), 0.f);
    __syncthreads();
    const int lane = j & 63, wave = j >> 6;
    for (int t = wave; t < R * kOut; t += 4) {
        const int r = t / kOut, o = t % kOut;
        float s = 0.f;
        for (int k = lane; k < kHidden; k += 64) s = fmaf(s_h2[r][k], bf16_to_f32(W3[k * kOut + o]), s);
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
        if (lane == 0 && r0 + r < P) Y[(size_t)(r0 + r) * kOut + o] = s + bf16_to_f32(B3[o]);
    }
}

constexpr uint32_t kFewRows = 1024;
static void launch_infer(hipStream_t s, uint32_t P, const uint8_t *state, const float *vsh, const float *esh,
                         const uint16_t *Wb, const uint16_t *Wi, float *Y) {
    if (P <= kFewRows) infer_kernel<2><<<(P + 1) / 2, 256, 0, s>>>(P, state, vsh, esh, Wb, Wi, Y);
    else infer_kernel<8><<<(P + 7) / 8, 256, 0, s>>>(P, state, vsh, esh, Wb, Wi, Y);
}

// A sequence number for the host, behind what the stream's kernels wrote to it.
static __global__ void infer_mark_kernel(uint32_t *flag, uint32_t seq) {
    __hip_atomic_store(flag, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---- host object ---------------------------------------------------------------
template <typename T>
static lt_status dalloc(T **p, size_t n) {
    if (hipMalloc((void **)p, sizeof(T) * (n ? n : 1)) != hipSuccess) {
        (void)hipGetLastError();
        set_error("hipMalloc of %zu bytes failed", sizeof(T) * n);
        return LT_E_NOMEM;
    }
    return LT_OK;
}

struct Scorer {
    uint32_t P = 0;
    hipStream_t stream = nullptr;
    float *d_vsh = nullptr, *d_esh = nullptr;
    std::vector<float> h_vsh, h_esh;
    float *W = nullptr, *Mo = nullptr, *Vo = nullptr;
    uint16_t *Wb = nullptr;
    uint16_t *Wi = nullptr;     // inference copy of W1, W2 (output-major)
    uint64_t wver = 0, wi_ver = ~0ull;  // bumped on every weight update; Wi is valid for wi_ver
    uint64_t uid = 0;                    // unique per scorer created in this process
    uint64_t adam_t = 0;
    bool trained = false;
    // training buffers (capacity in decisions)
    uint32_t cap = 0;
    uint8_t *h_batch = nullptr;  // a batch, pinned and mapped (see Batch)
    Batch batch{};               // device views of its arrays
    uint32_t *d_counts = nullptr;
    float *X = nullptr, *A1 = nullptr, *A2 = nullptr, *Y = nullptr, *dY = nullptr;
    float *small = nullptr, *w2 = nullptr;  // partial gradients
    float *d_losses = nullptr;              // per decision
    float *h_grad = nullptr, *d_grad = nullptr;  // pinned: the two losses, then the gradient
    // inference buffers
    uint8_t *h_stage = nullptr;  // one decision's packed state, pinned and mapped (see infer_kernel)
    float *h_Y = nullptr;        // its scores, written by the kernel into pinned mapped memory
    uint8_t *d_stage = nullptr;  // device views of h_stage and h_Y
    float *d_Y = nullptr;
    uint32_t infer_seq = 0;         // of the last launch, written behind h_Y's scores
    hipStream_t pending = nullptr;  // stream of the launched inference not yet waited for
    Samples data;

    ~Scorer();
    lt_status init(uint32_t P_, const uint32_t *node_off, const uint64_t *edge_off, uint64_t seed);
    lt_status ensure_cap(uint32_t n);
    lt_status forward_backward(uint32_t nb, bool update, float lr, bool grad_out);
    lt_status wait_infer();
};

Scorer::~Scorer() {
    if (pending) (void)hipStreamSynchronize(pending);
    if (stream) (void)hipStreamSynchronize(stream);
    void *ptrs[] = {d_vsh, d_esh, W, Mo, Vo, Wb, Wi, d_counts, X, A1, A2, Y, dY, small, w2, d_losses};
    for (void *p : ptrs)
        if (p) (void)hipFree(p);
    if (h_batch) (void)hipHostFree(h_batch);
    if (h_grad) (void)hipHostFree(h_grad);
    if (h_stage) (void)hipHostFree(h_stage);
    if (h_Y) (void)hipHostFree(h_Y);
    if (stream) (void)hipStreamDestroy(stream);
}

static std::atomic<uint64_t> g_scorer_uid{0};

lt_status Scorer::init(uint32_t P_, const uint32_t *node_off, const uint64_t *edge_off, uint64_t seed) {
    P = P_;
    uid = ++g_scorer_uid;
    MLP_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    const double V = std::max<double>(1.0, node_off[P]), E = std::max<double>(1.0, (double)edge_off[P]);
    h_vsh.resize(P);
    h_esh.resize(P);
    for (uint32_t q = 0; q < P; q++) {
        h_vsh[q] = (float)((node_off[q + 1] - node_off[q]) / V * P);
        h_esh[q] = (float)((edge_off[q + 1] - edge_off[q]) / E * P);
    }
    lt_status st;
    if ((st = dalloc(&d_vsh, P)) || (st = dalloc(&d_esh, P))) return st;
    MLP_HIP(hipMemcpy(d_vsh, h_vsh.data(), 4 * P, hipMemcpyHostToDevice));
    MLP_HIP(hipMemcpy(d_esh, h_esh.data(), 4 * P, hipMemcpyHostToDevice));
    if ((st = dalloc(&W, kParams)) || (st = dalloc(&Mo, kParams)) || (st = dalloc(&Vo, kParams)) ||
        (st = dalloc(&Wb, kParams)) || (st = dalloc(&Wi, kWiSize)))
        return st;
    // He-style initialisation from a seeded generator; biases zero.
    std::vector<float> w(kParams, 0.f);
    std::mt19937_64 rng(seed);
    auto fill = [&](size_t off, int fan_in, size_t n) {
        std::normal_distribution<float> nd(0.f, sqrtf(2.f / (float)fan_in));
        for (size_t i = 0; i < n; i++) w[off + i] = nd(rng);
    };
    fill(kOffW1, kFeat, (size_t)kFeat * kHidden);
    fill(kOffW2, kHidden, (size_t)kHidden * kHidden);
    fill(kOffW3, kHidden, (size_t)kHidden * kOut);
    for (size_t i = 0; i < (size_t)kHidden * kOut; i++) w[kOffW3 + i] *= 0.1f;
    MLP_HIP(hipMemcpy(W, w.data(), 4 * kParams, hipMemcpyHostToDevice));
    MLP_HIP(hipMemset(Mo, 0, 4 * kParams));
    MLP_HIP(hipMemset(Vo, 0, 4 * kParams));
    round_kernel<<<(kParams + 255) / 256, 256, 0, stream>>>(kParams, W, Wb);
    MLP_HIP(hipGetLastError());
    wver++;
    MLP_HIP(hipHostMalloc((void **)&h_stage, state_bytes(P), hipHostMallocMapped | hipHostMallocCoherent));
    const size_t y_bytes = sizeof(float) * P * kOut + 4;  // scores, sequence number
    MLP_HIP(hipHostMalloc((void **)&h_Y, y_bytes, hipHostMallocMapped | hipHostMallocCoherent));
    memset(h_Y, 0, y_bytes);
    MLP_HIP(hipHostGetDevicePointer((void **)&d_stage, h_stage, 0));
    MLP_HIP(hipHostGetDevicePointer((void **)&d_Y, h_Y, 0));
    MLP_HIP(hipStreamSynchronize(stream));
    return LT_OK;
}

// Buffers for batches of n decisions.  The batch's arrays lie one behind the
// other in pinned memory, which the forward and loss kernels read in place.
lt_status Scorer::ensure_cap(uint32_t n) {
    if (n <= cap) return LT_OK;
    cap = 0;
    for (void **p : {(void **)&d_counts, (void **)&X, (void **)&A1, (void **)&A2, (void **)&Y, (void **)&dY, (void **)&small,
                     (void **)&w2, (void **)&d_losses}) {
        if (*p) (void)hipFree(*p);
        *p = nullptr;
    }
    if (h_batch) (void)hipHostFree(h_batch);
    h_batch = nullptr;
    const size_t rows = (size_t)n * P, tiles = (rows + kTileRows - 1) / kTileRows;
    lt_status st;
    if ((st = dalloc(&d_counts, rows)) || (st = dalloc(&X, rows * kFeat)) || (st = dalloc(&A1, rows * kHidden)) ||
        (st = dalloc(&A2, rows * kHidden)) || (st = dalloc(&Y, rows * kOut)) || (st = dalloc(&dY, rows * kOut)) ||
        (st = dalloc(&small, std::min<size_t>(tiles, kGroupMost) * kSmallParams)) ||
        (st = dalloc(&w2, std::min<size_t>(tiles, kSliceMost) * kHidden * kHidden)) || (st = dalloc(&d_losses, 2 * (size_t)n)))
        return st;
    const size_t bytes = 13 * rows + (12 + 4 * kRecent + 16) * (size_t)n;
    MLP_HIP(hipHostMalloc((void **)&h_batch, bytes, hipHostMallocMapped | hipHostMallocCoherent));
    uint8_t *d = nullptr;
    MLP_HIP(hipHostGetDevicePointer((void **)&d, h_batch, 0));
    batch.counts = (const uint32_t *)d;
    batch.age = batch.counts + rows;
    batch.keep = (const float *)(batch.age + rows);
    batch.scale = batch.keep + rows;
    batch.recent = (const int32_t *)(batch.scale + 3 * (size_t)n);
    batch.cur = batch.recent + (size_t)n * kRecent;
    batch.next = batch.cur + n;
    batch.wa = (const float *)(batch.next + n);
    batch.wb = batch.wa + n;
    batch.resident = (const uint8_t *)(batch.wb + n);
    if (!h_grad) {
        MLP_HIP(hipHostMalloc((void **)&h_grad, 4 * (2 + kParams), hipHostMallocMapped | hipHostMallocCoherent));
        MLP_HIP(hipHostGetDevicePointer((void **)&d_grad, h_grad, 0));
    }
    cap = n;
    return LT_OK;
}

// Forward + backward over the nb decisions of the batch; h_grad receives the two
// losses and, with grad_out, the gradient; with update, one Adam step.
lt_status Scorer::forward_backward(uint32_t nb, bool update, float lr, bool grad_out) {
    const uint32_t M = nb * P, tiles = (M + kTileRows - 1) / kTileRows;
    const uint32_t groups = std::min(tiles, kGroupMost), slices = std::min(tiles, kSliceMost);
    hipStream_t s = stream;
    if (wi_ver != wver) {
        transpose_infer_weights_kernel<<<(unsigned)((kWiSize + 255) / 256), 256, 0, s>>>(Wb, Wi);
        wi_ver = wver;
    }
    train_forward_kernel<<<tiles, 256, 0, s>>>(P, M, batch, d_vsh, d_esh, Wb, Wi, d_counts, X, A1, A2, Y);
    loss_kernel<<<nb, 256, 0, s>>>(P, nb, Y, d_counts, batch.next, batch.keep, batch.wa, batch.wb, dY, d_losses);
    train_backward_kernel<<<groups + 4 * slices, 256, 0, s>>>(M, groups, slices, X, A1, A2, dY, Wb, small, w2);
    float b1t = 0.f, b2t = 0.f;
    if (update) {
        adam_t++;
        b1t = powf(0.9f, (float)adam_t);
        b2t = powf(0.999f, (float)adam_t);
        wi_ver = ++wver;  // the update writes Wi as well
    }
    train_update_kernel<<<(unsigned)((kParams + 31) / 32), 256, 0, s>>>(groups, slices, small, w2,
                                                                       grad_out ? d_grad + 2 : nullptr, W, Wb, Wi, Mo, Vo,
                                                                       update ? 1 : 0, lr, b1t, b2t, nb, d_losses, d_grad);
    MLP_HIP(hipGetLastError());
    return LT_OK;
}

Scorer *scorer_new(uint32_t P, const uint32_t *node_off, const uint64_t *edge_off, uint64_t seed, lt_status *st) {
    std::unique_ptr<Scorer> s(new Scorer);
    *st = s->init(P, node_off, edge_off, seed);
    if (*st != LT_OK) return nullptr;
    return s.release();
}

void scorer_free(Scorer *s) { delete s; }
Samples &scorer_samples(Scorer *s) { return s->data; }
uint32_t scorer_partitions(const Scorer *s) { return s->P; }
bool scorer_trained(const Scorer *s) { return s && s->trained; }

// Stage one decision's state in pinned mapped memory in the packed layout of
// infer_kernel, which reads it over the bus, and launch the fused MLP on
// `stream` (nullptr = the scorer's own); scorer_infer_wait returns the scores,
// which come back the same way.  A launch first waits for the one before it,
// whose kernel may still be reading the staged state.
lt_status scorer_infer_launch(Scorer *s, const DecisionState &d, void *stream_v) {
    hipStream_t st = stream_v ? (hipStream_t)stream_v : s->stream;
    lt_status rc = s->wait_infer();
    if (rc != LT_OK) return rc;
    const uint32_t P = s->P;
    uint8_t *h = s->h_stage;
    pack_state_head((int32_t *)h, d.counts, P, d.recent, d.cur, d.w_total);
    memcpy(h + kStateHead, d.counts, 4 * (size_t)P);
    memcpy(h + kStateHead + 4 * (size_t)P, d.age, 4 * (size_t)P);
    memcpy(h + kStateHead + 8 * (size_t)P, d.resident, P);
    if (s->wi_ver != s->wver) {
        transpose_infer_weights_kernel<<<(unsigned)((kWiSize + 255) / 256), 256, 0, st>>>(s->Wb, s->Wi);
        MLP_HIP(hipGetLastError());
        s->wi_ver = s->wver;
    }
    launch_infer(st, P, s->d_stage, s->d_vsh, s->d_esh, s->Wb, s->Wi, s->d_Y);
    infer_mark_kernel<<<1, 1, 0, st>>>((uint32_t *)(s->d_Y + (size_t)P * kOut), ++s->infer_seq);
    MLP_HIP(hipGetLastError());
    s->pending = st;
    return LT_OK;
}

// The last launched inference is over: its sequence number is there.  Polled in
// memory; the stream itself is asked only once in a while.
lt_status Scorer::wait_infer() {
    if (!pending) return LT_OK;
    const hipStream_t st = pending;
    pending = nullptr;
    const uint32_t *flag = (const uint32_t *)(h_Y + (size_t)P * kOut);
    for (uint32_t it = 1; __atomic_load_n(flag, __ATOMIC_ACQUIRE) != infer_seq; it++) {
        __builtin_ia32_pause();
        if ((it & 0xFFFFF) == 0) {
            const hipError_t e = hipStreamQuery(st);
            if (e == hipErrorNotReady) continue;
            MLP_HIP(e);
            if (__atomic_load_n(flag, __ATOMIC_ACQUIRE) == infer_seq) break;
            set_error("scores were not written");
            return LT_E_INTERNAL;
        }
    }
    return LT_OK;
}

// Scores (out[P*2]) of the last launched inference.  Polls: this wait can be
// on the scheduler's critical path.
lt_status scorer_infer_wait(Scorer *s, float *out) {
    if (!s->pending) {
        set_error("no inference in flight");
        return LT_E_INTERNAL;
    }
    lt_status st = s->wait_infer();
    if (st != LT_OK) return st;
    memcpy(out, s->h_Y, sizeof(float) * s->P * kOut);
    return LT_OK;
}

bool scorer_infer_pending(const Scorer *s) { return s && s->pending; }

lt_status scorer_infer(Scorer *s, const DecisionState &d, void *stream_v, float *out) {
    lt_status st = scorer_infer_launch(s, d, stream_v);
    return st != LT_OK ? st : scorer_infer_wait(s, out);
}

// ---- inference without allocation ----------------------------------------------
// Scratch of lt_scorer_infer_noalloc, one copy per GPU, held until the
// process ends: one decision's packed state (the layout infer_kernel reads),
// its scores, and the output-major copy of the first two layers' weights.
// Sized for kNoAllocMaxP partitions (about 1.4 MB).  In host code the name
// `scratch` is only a stand-in for the symbol: its device address comes from
// hipGetSymbolAddress, once per device, and only that address is used.
constexpr uint32_t kNoAllocMaxP = 65535;  // the largest partition count a .part file holds
constexpr size_t kNaStateBytes = (state_bytes(kNoAllocMaxP) + 255) & ~(size_t)255;
constexpr size_t kNaYBytes = ((sizeof(float) * kNoAllocMaxP * kOut) + 255) & ~(size_t)255;
constexpr size_t kNaWiBytes = ((sizeof(uint16_t) * kWiSize) + 255) & ~(size_t)255;
static __device__ __align__(256) uint8_t scratch[kNaStateBytes + kNaYBytes + kNaWiBytes];

namespace {
constexpr int kNaMaxDevices = 64;
struct NoAllocDevice {
    uint8_t *base = nullptr;          // device address of this GPU's scratch
    uint64_t wi_uid = 0;  // scorer (Scorer::uid) whose weights the scratch's inference copy holds
    uint64_t wi_ver = 0;  // and their version
};
NoAllocDevice g_noalloc[kNaMaxDevices];
std::mutex g_noalloc_mu;
}  // namespace

// This GPU's scratch address, looked up on the first call made on it.
static lt_status noalloc_scratch(int dev, NoAllocDevice **out) {
    if (dev < 0 || dev >= kNaMaxDevices) {
        set_error("lt_scorer_infer_noalloc: device %d beyond the %d supported", dev, kNaMaxDevices);
        return LT_E_ARG;
    }
    std::lock_guard<std::mutex> lock(g_noalloc_mu);
    NoAllocDevice &d = g_noalloc[dev];
    if (!d.base) {
        void *ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) {
            set_error("lt_scorer_infer_noalloc: hipGetSymbolAddress(scratch) on device %d: %s", dev,
                      hipGetErrorString(e));
            return LT_E_HIP;
        }
        d.base = (uint8_t *)ptr;
    }
    *out = &d;
    return LT_OK;
}

}  // namespace lt

struct lt_scorer : lt::Scorer {};

using namespace lt;

// Writes decisions off .. off + nb (or order[off ..]) to the pinned batch; the
// step before, which reads it, is over.
static void stage_batch(Scorer *s, uint64_t off, uint32_t nb, const uint32_t *counts, const uint8_t *resident,
                        const uint32_t *age, const int32_t *recent, const int32_t *cur, const float *w_total,
                        const int32_t *next_label, const float *keep_label, const float *wa, const float *wb,
                        const std::vector<uint64_t> *order) {
    const size_t P = s->P;
    const auto at = [&](const void *p) { return s->h_batch + ((const uint8_t *)p - (const uint8_t *)s->batch.counts); };
    uint32_t *c = (uint32_t *)at(s->batch.counts), *ag = (uint32_t *)at(s->batch.age);
    float *kp = (float *)at(s->batch.keep), *sc = (float *)at(s->batch.scale);
    int32_t *rc = (int32_t *)at(s->batch.recent), *cu = (int32_t *)at(s->batch.cur), *nx = (int32_t *)at(s->batch.next);
    float *a = (float *)at(s->batch.wa), *b = (float *)at(s->batch.wb);
    uint8_t *r = at(s->batch.resident);
    for (size_t i = 0; i < nb; i++) {
        const uint64_t j = order ? (*order)[off + i] : off + i;
        memcpy(c + i * P, counts + j * P, 4 * P);
        memcpy(r + i * P, resident + j * P, P);
        memcpy(ag + i * P, age + j * P, 4 * P);
        memcpy(rc + i * kRecent, recent + j * kRecent, 4 * kRecent);
        cu[i] = cur[j];
        nx[i] = next_label[j];
        uint32_t mx = 0;
        uint64_t sum = 0;
        for (size_t q = 0; q < P; q++) {
            mx = std::max(mx, counts[j * P + q]);
            sum += counts[j * P + q];
        }
        sc[3 * i] = w_total[j];
        sc[3 * i + 1] = (float)mx;
        sc[3 * i + 2] = (float)sum;
        if (keep_label) memcpy(kp + i * P, keep_label + j * P, 4 * P);
        else memset(kp + i * P, 0, 4 * P);
        a[i] = wa ? wa[j] : 1.f;
        b[i] = (wb && keep_label) ? wb[j] : 0.f;
    }
}

extern "C" {

lt_status lt_scorer_create(const lt_partition *p, uint64_t seed, lt_scorer **out) {
    if (!p || !out) return LT_E_ARG;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n == 0) {
        (void)hipGetLastError();
        set_error("the scorer needs a HIP device");
        return LT_E_NODEVICE;
    }
    std::unique_ptr<lt_scorer> s(new lt_scorer);
    lt_status st = s->init(p->P(), p->node_off.data(), p->edge_off.data(), seed);
    if (st != LT_OK) return st;
    *out = s.release();
    return LT_OK;
}

void lt_scorer_free(lt_scorer *s) { delete s; }

lt_status lt_scorer_loss_grad(lt_scorer *s, uint64_t n, const uint32_t *counts, const uint8_t *resident,
                              const uint32_t *age, const int32_t *recent, const int32_t *cur, const float *w_total,
                              const int32_t *next_label, const float *keep_label, const float *wa, const float *wb,
                              float *loss_out, float *grad_out) {
    if (!s || !n || !counts || !resident || !age || !recent || !cur || !w_total || !next_label) return LT_E_ARG;
    if (n > 512) {
        set_error("at most 512 decisions per call");
        return LT_E_ARG;
    }
    lt_status st = s->ensure_cap((uint32_t)n);
    if (st != LT_OK) return st;
    stage_batch(s, 0, (uint32_t)n, counts, resident, age, recent, cur, w_total, next_label, keep_label, wa, wb, nullptr);
    if ((st = s->forward_backward((uint32_t)n, false, 0.f, grad_out != nullptr)) != LT_OK) return st;
    MLP_HIP(hipStreamSynchronize(s->stream));
    if (loss_out) memcpy(loss_out, s->h_grad, 8);
    if (grad_out) memcpy(grad_out, s->h_grad + 2, 4 * kParams);
    return LT_OK;
}

lt_status lt_scorer_train(lt_scorer *s, uint64_t n, const uint32_t *counts, const uint8_t *resident,
                          const uint32_t *age, const int32_t *recent, const int32_t *cur, const float *w_total,
                          const int32_t *next_label, const float *keep_label, const float *wa, const float *wb,
                          uint32_t epochs, uint32_t batch, float lr, uint64_t seed, float *loss_out) {
    if (!s || !n || !counts || !resident || !age || !recent || !cur || !w_total || !next_label || !batch || !epochs)
        return LT_E_ARG;
    batch = std::min<uint32_t>(batch, (uint32_t)std::min<uint64_t>(n, 512));
    lt_status st = s->ensure_cap(batch);
    if (st != LT_OK) return st;
    std::vector<uint64_t> order(n);
    for (uint64_t i = 0; i < n; i++) order[i] = i;
    std::mt19937_64 rng(seed);
    float last[2] = {0, 0};
    for (uint32_t e = 0; e < epochs; e++) {
        std::shuffle(order.begin(), order.end(), rng);
        double acc[2] = {0, 0};
        uint32_t steps = 0;
        for (uint64_t off = 0; off + batch <= n; off += batch) {
            stage_batch(s, off, batch, counts, resident, age, recent, cur, w_total, next_label, keep_label, wa, wb, &order);
            if ((st = s->forward_backward(batch, true, lr, false)) != LT_OK) return st;
            MLP_HIP(hipStreamSynchronize(s->stream));
            const float *l = s->h_grad;
            acc[0] += l[0];
            acc[1] += l[1];
            steps++;
        }
        if (steps) {
            last[0] = (float)(acc[0] / steps);
            last[1] = (float)(acc[1] / steps);
        }
    }
    for (int i = 0; i < 2; i++)
        if (!std::isfinite(last[i])) {
            set_error("scorer training diverged");
            return LT_E_INTERNAL;
        }
    s->trained = true;
    if (loss_out) {
        loss_out[0] = last[0];
        loss_out[1] = last[1];
    }
    return LT_OK;
}

lt_status lt_scorer_infer(lt_scorer *s, const uint32_t *counts, const uint8_t *resident, const uint32_t *age,
                          const int32_t *recent, int32_t cur, float w_total, float *out) {
    if (!s || !counts || !resident || !age || !recent || !out) return LT_E_ARG;
    DecisionState d;
    d.counts = counts;
    d.resident = resident;
    d.age = age;
    for (int k = 0; k < kRecent; k++) d.recent[k] = recent[k];
    d.cur = cur;
    d.w_total = w_total;
    return scorer_infer(s, d, s->stream, out);
}

// The scores of lt_scorer_infer, computed through the GPU's static scratch
// instead of the scorer's staging buffers: state copied in, infer_kernel,
// scores copied out, all on the scorer's stream; no allocation of any kind.
lt_status lt_scorer_infer_noalloc(lt_scorer *s, const uint32_t *counts, const uint8_t *resident, const uint32_t *age,
                                  const int32_t *recent, int32_t cur, float w_total, float *out) {
    if (!s || !counts || !resident || !age || !recent || !out) return LT_E_ARG;
    const uint32_t P = s->P;
    if (P > kNoAllocMaxP) {
        set_error("lt_scorer_infer_noalloc: %u partitions exceed the scratch's %u", P, kNoAllocMaxP);
        return LT_E_ARG;
    }
    int dev = 0;
    MLP_HIP(hipGetDevice(&dev));
    NoAllocDevice *nd = nullptr;
    LT_NA_TRY(noalloc_scratch(dev, &nd));
    uint8_t *state = nd->base, *Y = nd->base + kNaStateBytes, *Wi = nd->base + kNaStateBytes + kNaYBytes;
    int32_t head[kStateHead / 4];
    pack_state_head(head, counts, P, recent, cur, w_total);
    hipStream_t st = s->stream;
    MLP_HIP(hipMemcpyAsync(state, head, kStateHead, hipMemcpyHostToDevice, st));
    MLP_HIP(hipMemcpyAsync(state + kStateHead, counts, 4 * (size_t)P, hipMemcpyHostToDevice, st));
    MLP_HIP(hipMemcpyAsync(state + kStateHead + 4 * (size_t)P, age, 4 * (size_t)P, hipMemcpyHostToDevice, st));
    MLP_HIP(hipMemcpyAsync(state + kStateHead + 8 * (size_t)P, resident, P, hipMemcpyHostToDevice, st));
    {
        std::lock_guard<std::mutex> lock(g_noalloc_mu);
        if (nd->wi_uid != s->uid || nd->wi_ver != s->wver) {  // the scratch holds other weights
            transpose_infer_weights_kernel<<<(unsigned)((kWiSize + 255) / 256), 256, 0, st>>>(s->Wb,
                                                                                              (uint16_t *)Wi);
            MLP_HIP(hipGetLastError());
            nd->wi_uid = s->uid;
            nd->wi_ver = s->wver;
        }
    }
    launch_infer(st, P, state, s->d_vsh, s->d_esh, s->Wb, (const uint16_t *)Wi, (float *)Y);
    MLP_HIP(hipGetLastError());
    MLP_HIP(hipMemcpyAsync(out, Y, sizeof(float) * P * kOut, hipMemcpyDeviceToHost, st));
    MLP_HIP(hipStreamSynchronize(st));
    return LT_OK;
}

uint64_t lt_scorer_num_params(void) { return kParams; }

lt_status lt_scorer_fit(lt_scorer *s, uint32_t epochs, uint32_t batch, float lr, uint64_t seed, float *loss_out) {
    if (!s) return LT_E_ARG;
    Samples &d = s->data;
    if (d.n == 0) {
        set_error("no training samples: add traces first");
        return LT_E_ARG;
    }
    return lt_scorer_train(s, d.n, d.counts.data(), d.resident.data(), d.age.data(), d.recent.data(), d.cur.data(),
                           d.w_total.data(), d.next.data(), d.keep.data(), d.wa.data(), d.wb.data(), epochs, batch, lr,
                           seed, loss_out);
}

lt_status lt_scorer_get_params(const lt_scorer *s, float *out) {
    if (!s || !out) return LT_E_ARG;
    MLP_HIP(hipMemcpy(out, s->W, 4 * kParams, hipMemcpyDeviceToHost));
    return LT_OK;
}

lt_status lt_scorer_set_params(lt_scorer *s, const float *in) {
    if (!s || !in) return LT_E_ARG;
    MLP_HIP(hipMemcpy(s->W, in, 4 * kParams, hipMemcpyHostToDevice));
    round_kernel<<<(kParams + 255) / 256, 256, 0, s->stream>>>(kParams, s->W, s->Wb);
    MLP_HIP(hipGetLastError());
    s->wver++;
    MLP_HIP(hipStreamSynchronize(s->stream));
    s->trained = true;
    return LT_OK;
}

// File: "LTMLP2\0\0" | u32 features | u32 hidden | u32 outputs | u32 pad | u16 bf16 weights[kParams]
lt_status lt_scorer_save(const lt_scorer *s, const char *path) {
    if (!s || !path) return LT_E_ARG;
    std::vector<uint16_t> wb(kParams);
    MLP_HIP(hipMemcpy(wb.data(), s->Wb, 2 * kParams, hipMemcpyDeviceToHost));
    FILE *f = fopen(path, "wb");
    if (!f) {
        set_error("cannot create %s", path);
        return LT_E_IO;
    }
    const char magic[8] = {'L', 'T', 'M', 'L', 'P', '2', 0, 0};
    const uint32_t hdr[4] = {kFeat, kHidden, kOut, 0};
    bool ok = fwrite(magic, 1, 8, f) == 8 && fwrite(hdr, 4, 4, f) == 4 && fwrite(wb.data(), 2, kParams, f) == kParams;
    ok = fclose(f) == 0 && ok;
    if (!ok) {
        set_error("write to %s failed", path);
        return LT_E_IO;
    }
    return LT_OK;
}

lt_status lt_scorer_load(lt_scorer *s, const char *path) {
    if (!s || !path) return LT_E_ARG;
    FILE *f = fopen(path, "rb");
    if (!f) {
        set_error("cannot open %s", path);
        return LT_E_IO;
    }
    char magic[8];
    uint32_t hdr[4];
    std::vector<uint16_t> wb(kParams);
    bool ok = fread(magic, 1, 8, f) == 8 && fread(hdr, 4, 4, f) == 4 && fread(wb.data(), 2, kParams, f) == kParams;
    fclose(f);
    if (!ok || memcmp(magic, "LTMLP2", 6) != 0 || hdr[0] != kFeat || hdr[1] != kHidden || hdr[2] != kOut) {
        set_error("%s is not a scorer weights file", path);
        return LT_E_FORMAT;
    }
    std::vector<float> w(kParams);
    for (size_t i = 0; i < kParams; i++) {
        const uint32_t u = (uint32_t)wb[i] << 16;
        memcpy(&w[i], &u, 4);
    }
    return lt_scorer_set_params(s, w.data());
}

}  // extern "C"
