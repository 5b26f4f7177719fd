// The learned pruner's network: an MLP 64 -> 128 -> 128 -> 1 (ReLU, ReLU,
// logit), bf16 weights with fp32 accumulation, and its training (weighted
// binary cross-entropy, Adam on fp32 master weights that are rounded to bf16
// after every step, so the forward pass always sees the bf16 weights).
//
// Parameters, packed (kMlpParams values; the bf16 copy has the same layout):
//   W1 [128][64] | b1 [128] | W2 [128][128] | b2 [128] | w3 [128] | b3 [1]
//
// Both layers run on the matrix cores.  The forward pass multiplies bf16
// weights with float32 activations exactly: an activation is the sum of three
// bf16 values (8 + 8 + 8 bits of its significand, cut off, no rounding), each
// product of two bf16 values is exact in float32, and only the sums round, as
// in a float32 chain.  The gradient's products of two float32 values use the
// float32 matrix instructions.  Every sum runs in a fixed order (the gradient
// per block over its tiles and then over the blocks, k_mlp_reduce), so results
// do not depend on timing.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "inscy_internal.h"

#pragma clang fp contract(off)

namespace inscy {

namespace {

constexpr int kIn = kMlpIn, kH = kMlpHidden;
constexpr int kThreads = 256;
constexpr int kTile = 32;             // samples per tile
constexpr int kHalf = kTile / 2;      // samples per thread in the layer passes
constexpr int kW1 = 0, kB1 = kW1 + kH * kIn, kW2 = kB1 + kH, kB2 = kW2 + kH * kH, kW3 = kB2 + kH, kB3 = kW3 + kH;
static_assert(kB3 + 1 == kMlpParams, "parameter layout");
static_assert(kThreads == 2 * kH, "two threads per hidden unit");

__device__ __forceinline__ float bf16_to_f32(uint16_t h) { return __uint_as_float((uint32_t) h << 16); }

// round to nearest even (finite inputs)
__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
    const uint32_t u = __float_as_uint(f);
    const uint32_t r = 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t) ((u + r) >> 16);
}

// a tile of the VALU forward pass
struct Tile {
    float x[kTile][kIn];
    float h1[kTile][kH];
    float h2[kTile][kH];
    float z[kTile];
};

__device__ void load_tile(const float *__restrict__ X, long long N, long long t0, Tile &T, int &ns) {
    ns = (int) min((long long) kTile, N - t0);
    for (int e = threadIdx.x; e < kTile * kIn; e += blockDim.x) {
        const int s = e / kIn, i = e % kIn;
        T.x[s][i] = s < ns ? X[(t0 + s) * kIn + i] : 0.0f;
    }
    __syncthreads();
}

// out[s][j] = relu(b[j] + sum_i in[s][i] W[j][i]) for the thread's unit j and
// its half of the tile's samples
template <int K>
__device__ __forceinline__ void layer(const uint16_t *__restrict__ W, const uint16_t *__restrict__ b,
                                      const float (*in)[K], float (*out)[kH], int ns) {
    const int j = threadIdx.x & (kH - 1), s0 = (threadIdx.x >> 7) * kHalf;
    float acc[kHalf];
    const float bj = bf16_to_f32(b[j]);
#pragma unroll
    for (int s = 0; s < kHalf; ++s) acc[s] = bj;
    for (int i0 = 0; i0 < K; i0 += 8) {
        float w[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) w[u] = bf16_to_f32(W[j * K + i0 + u]);
#pragma unroll
        for (int s = 0; s < kHalf; ++s)
#pragma unroll
            for (int u = 0; u < 8; ++u) acc[s] = fmaf(in[s0 + s][i0 + u], w[u], acc[s]);
    }
#pragma unroll
    for (int s = 0; s < kHalf; ++s) out[s0 + s][j] = s0 + s < ns ? fmaxf(acc[s], 0.0f) : 0.0f;
}

// The tile through the network: h1, h2 (after ReLU) and the logits z.
__device__ void tile_forward(const uint16_t *__restrict__ P, Tile &T, int ns) {
    layer<kIn>(P + kW1, P + kB1, T.x, T.h1, ns);
    __syncthreads();
    layer<kH>(P + kW2, P + kB2, T.h1, T.h2, ns);
    __syncthreads();
    // logits: 8 consecutive lanes per sample, 16 terms each, then a fixed
    // butterfly over the 8 lanes
    {
        const int s = threadIdx.x >> 3, q = threadIdx.x & 7;
        float acc = 0.0f;
        for (int i = q * 16; i < q * 16 + 16; ++i) acc = fmaf(T.h2[s][i], bf16_to_f32(P[kW3 + i]), acc);
        acc += __shfl_xor(acc, 1);
        acc += __shfl_xor(acc, 2);
        acc += __shfl_xor(acc, 4);
        if (q == 0) T.z[s] = acc + bf16_to_f32(P[kB3]);
    }
    __syncthreads();
}

// ------------------------------------------------------------ forward pass on bf16 matrix cores
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
// the caller's arrays: samples at least 4-byte, parameters 2-byte aligned
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t param4 __attribute__((ext_vector_type(2), aligned(2)));  // 4 parameters
__device__ __forceinline__ uint2 load_param4(const uint16_t *p) {
    const param4 v = *reinterpret_cast<const param4 *>(p);
    return make_uint2(v.x, v.y);
}

// x = hi + mid + lo exactly, three bf16 values in the upper halves of words
// (an infinity or NaN is its own hi)
__device__ __forceinline__ void split3(float x, uint32_t &hi, uint32_t &mid, uint32_t &lo) {
    const uint32_t u = __float_as_uint(x);
    const bool fin = (u & 0x7F800000u) != 0x7F800000u;
    hi = (u & 0xFFFF0000u) | ((u & 0x7FFFFFFFu) > 0x7F800000u ? 0x00400000u : 0u);
    const float r1 = fin ? x - __uint_as_float(hi) : 0.0f;
    mid = __float_as_uint(r1) & 0xFFFF0000u;
    lo = __float_as_uint(r1 - __uint_as_float(mid));
}
struct Split8 {
    bf16x8 p[3];
};
__device__ __forceinline__ Split8 split8(const float (&v)[8]) {
    uint32_t w[3][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        uint32_t a[3], b[3];
        split3(v[2 * j], a[0], a[1], a[2]);
        split3(v[2 * j + 1], b[0], b[1], b[2]);
#pragma unroll
        for (int q = 0; q < 3; ++q) w[q][j] = (a[q] >> 16) | (b[q] & 0xFFFF0000u);
    }
    Split8 s;
#pragma unroll
    for (int q = 0; q < 3; ++q) s.p[q] = __builtin_bit_cast(bf16x8, make_uint4(w[q][0], w[q][1], w[q][2], w[q][3]));
    return s;
}

// Scores of 32 samples per wave, hidden units by samples: D = W B + bias with
// v_mfma_f32_32x32x16_bf16, three instructions (lo, mid, hi) per 16 inputs.
// Lane l holds sample l % 32; of a 32-unit tile of D it holds the units
// 8 q + 4 (l / 32) + i, and the second layer takes its inputs in exactly that
// order (its weights are laid out to match), so activations stay in registers.
// The weights lie in LDS in operand order (16 bytes a lane, no bank conflicts),
// loaded once per block; the blocks walk the tiles.
// 200,003 rows: 695 us with VALU sums, 41 now alone and 35 among others; bound by the
// matrix cores (144 instructions a tile) and the activation splits, at two waves
// per SIMD.
constexpr int kMfTiles = kH / 32;         // 32-unit tiles of a layer
constexpr int kK1 = kIn / 16, kK2 = kH / 16;  // 16-input steps
struct PredictLds {
    uint4 w1[kMfTiles * kK1][64];
    uint4 w2[kMfTiles * kK2][64];
    float b1[kH], b2[kH], w3[kH];
};
__global__ __launch_bounds__(kThreads) void k_mlp_predict(const float *__restrict__ X, long long N,
                                                          const uint16_t *__restrict__ P, float *__restrict__ prob) {
    __shared__ union {
        PredictLds m;
        Tile t;
    } L;
    // operand order; a weight that is not finite (it would spoil the split's
    // zero parts) sends the block to the plain pass
    bool bad = false;
    auto scan = [&](uint2 v) {
        const uint32_t e = 0x7F80u;
        bad |= (v.x & e) == e || ((v.x >> 16) & e) == e || (v.y & e) == e || ((v.y >> 16) & e) == e;
    };
    for (int i = threadIdx.x; i < kMfTiles * kK1 * 64; i += kThreads) {
        const int l = i & 63, c = (i >> 6) % kK1, t = (i >> 6) / kK1;
        const int at = kW1 + (32 * t + (l & 31)) * kIn + 16 * c + 8 * (l >> 5);
        const uint2 a = load_param4(P + at), b = load_param4(P + at + 4);
        scan(a);
        scan(b);
        L.m.w1[t * kK1 + c][l] = make_uint4(a.x, a.y, b.x, b.y);
    }
    for (int i = threadIdx.x; i < kMfTiles * kK2 * 64; i += kThreads) {
        const int l = i & 63, c = (i >> 6) % kK2, t = (i >> 6) / kK2;
        const int at = kW2 + (32 * t + (l & 31)) * kH + 16 * c + 4 * (l >> 5);
        const uint2 a = load_param4(P + at), b = load_param4(P + at + 8);
        scan(a);
        scan(b);
        L.m.w2[t * kK2 + c][l] = make_uint4(a.x, a.y, b.x, b.y);
    }
    if (threadIdx.x < kH) {
        L.m.b1[threadIdx.x] = bf16_to_f32(P[kB1 + threadIdx.x]);
        L.m.b2[threadIdx.x] = bf16_to_f32(P[kB2 + threadIdx.x]);
        L.m.w3[threadIdx.x] = bf16_to_f32(P[kW3 + threadIdx.x]);
    }
    const float b3 = bf16_to_f32(P[kB3]);
    if (__syncthreads_or(bad)) {
        for (long long t0 = (long long) blockIdx.x * kTile; t0 < N; t0 += (long long) gridDim.x * kTile) {
            int ns;
            load_tile(X, N, t0, L.t, ns);
            tile_forward(P, L.t, ns);
            if ((int) threadIdx.x < ns) prob[t0 + threadIdx.x] = 1.0f / (1.0f + expf(-L.t.z[threadIdx.x]));
            __syncthreads();
        }
        return;
    }
    const int l = __lane_id(), n = l & 31, h = l >> 5;
    const long long tiles = (N + 31) / 32;
    const long long step = (long long) gridDim.x * (kThreads / 64);
    for (long long tl = (long long) blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6); tl < tiles; tl += step) {
        // what the tiles share is read again in each (from LDS): held in
        // registers it would leave one wave per SIMD
        asm volatile("" ::: "memory");
        const long long row = min(tl * 32 + n, N - 1);
        const float *x = X + row * kIn + 8 * h;
        float xv[kK1][8];
#pragma unroll
        for (int c = 0; c < kK1; ++c) {
            const f32x4u a = *reinterpret_cast<const f32x4u *>(x + 16 * c);
            const f32x4u b = *reinterpret_cast<const f32x4u *>(x + 16 * c + 4);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                xv[c][j] = a[j];
                xv[c][4 + j] = b[j];
            }
        }
        f32x16 a1[kMfTiles];
#pragma unroll
        for (int t = 0; t < kMfTiles; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const f32x4 b = *reinterpret_cast<const f32x4 *>(&L.m.b1[32 * t + 8 * q + 4 * h]);
#pragma unroll
                for (int r = 0; r < 4; ++r) a1[t][4 * q + r] = b[r];
            }
#pragma unroll
        for (int c = 0; c < kK1; ++c) {
            const Split8 s = split8(xv[c]);
#pragma unroll
            for (int t = 0; t < kMfTiles; ++t) {
                const bf16x8 w = __builtin_bit_cast(bf16x8, L.m.w1[t * kK1 + c][l]);
#pragma unroll
                for (int q = 2; q >= 0; --q) a1[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, s.p[q], a1[t], 0, 0, 0);
            }
        }
        asm volatile("" ::: "memory");
        f32x16 a2[kMfTiles];
#pragma unroll
        for (int t = 0; t < kMfTiles; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const f32x4 b = *reinterpret_cast<const f32x4 *>(&L.m.b2[32 * t + 8 * q + 4 * h]);
#pragma unroll
                for (int r = 0; r < 4; ++r) a2[t][4 * q + r] = b[r];
            }
#pragma unroll
        for (int c = 0; c < kK2; ++c) {
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = fmaxf(a1[c >> 1][8 * (c & 1) + j], 0.0f);
            const Split8 s = split8(v);
#pragma unroll
            for (int t = 0; t < kMfTiles; ++t) {
                const bf16x8 w = __builtin_bit_cast(bf16x8, L.m.w2[t * kK2 + c][l]);
#pragma unroll
                for (int q = 2; q >= 0; --q) a2[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, s.p[q], a2[t], 0, 0, 0);
            }
        }
        float z[kMfTiles];
#pragma unroll
        for (int t = 0; t < kMfTiles; ++t) {
            z[t] = 0.0f;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const f32x4 w = *reinterpret_cast<const f32x4 *>(&L.m.w3[32 * t + 8 * q + 4 * h]);
#pragma unroll
                for (int r = 0; r < 4; ++r) z[t] = fmaf(fmaxf(a2[t][4 * q + r], 0.0f), w[r], z[t]);
            }
        }
        float zz = (z[0] + z[1]) + (z[2] + z[3]);
        zz += __shfl_xor(zz, 32);
        zz += b3;
        if (h == 0 && tl * 32 + n < N) prob[tl * 32 + n] = 1.0f / (1.0f + expf(-zz));
    }
}

// ------------------------------------------------------------ gradient on float32 matrix cores
// Gradient of  inv_wsum * sum_s wt_s * (softplus(z_s) - y_s z_s)  over the
// samples of this block's tiles, written to this block's row of `part`
// ([gridDim.x][kMlpParams + 1], the last column the loss).
// A block takes 32 samples at a time through 16 waves.  Every product is a
// 16 x 16 tile of v_mfma_f32_16x16x4_f32 per wave: the layers and the error at
// layer 1 as (8 unit tiles x 2 sample tiles), the weight gradients (sums over
// the 32 samples) as 4 tiles of dW2 and 2 of dW1 per wave, kept in registers
// over the block's tiles.  The minibatch's tiles fill half the CUs at most, so
// the time is the chain of one tile: 4,096 rows 114 us with VALU sums by 4 waves,
// 24 now, alone (a step with the reduction and Adam 26 among others).
constexpr int kGradThreads = 1024;
constexpr int kXs = kIn + 4, kHs = kH + 4;  // padded rows (LDS banks)
constexpr int kWs = kH + 16;
struct alignas(16) GradLds {
    float x[kTile][kXs];
    float h1[kTile][kHs];
    float h2[kTile][kHs];  // after the error at layer 2 is formed: the error at layer 1
    float d2[kTile][kHs];
    uint16_t w2[kH][kWs];
    float z[kTile], dz[kTile];
};

__global__ __launch_bounds__(kGradThreads) void k_mlp_grad(const float *__restrict__ X, const float *__restrict__ Y,
                                                           const float *__restrict__ WT, long long N, float inv_wsum,
                                                           const uint16_t *__restrict__ P, float *__restrict__ part) {
    __shared__ GradLds T;
    const int t = threadIdx.x, l = __lane_id(), wv = t >> 6;
    const int li = l & 15, lk = l >> 4;           // row / column of an operand, its quarter of the inputs
    const int ut = wv >> 1, st = wv & 1;          // layer passes: unit tile, sample tile
    const int unit = 16 * ut + li, smp = 16 * st + li;
    for (int e = t; e < kH * kH / 4; e += kGradThreads) {
        const int j = e / (kH / 4), c = e % (kH / 4);
        *reinterpret_cast<uint2 *>(&T.w2[j][4 * c]) = load_param4(P + kW2 + 4 * e);
    }
    f32x4 g2[4], g1[2];  // dW2 tiles 4 wv .. 4 wv + 3 (row-major over 8 x 8), dW1 tiles 2 wv, 2 wv + 1 (8 x 4)
#pragma unroll
    for (int q = 0; q < 4; ++q) g2[q] = f32x4{0.f, 0.f, 0.f, 0.f};
    g1[0] = g1[1] = f32x4{0.f, 0.f, 0.f, 0.f};
    float gsum = 0.0f;              // threads 0..383: gw3, gb2, gb1 of unit t % 128
    float gb3 = 0.0f, lsum = 0.0f;  // threads 0..31: their sample slot
    for (long long t0 = (long long) blockIdx.x * kTile; t0 < N; t0 += (long long) gridDim.x * kTile) {
        const int ns = (int) min((long long) kTile, N - t0);
        for (int e = t; e < kTile * kIn; e += kGradThreads) {
            const int s = e / kIn, i = e % kIn;
            T.x[s][i] = s < ns ? X[(t0 + s) * kIn + i] : 0.0f;
        }
        __syncthreads();
        // layer 1: inputs 16 lk + k, k = 0..15
        {
            f32x4 acc;
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[r] = bf16_to_f32(P[kB1 + 16 * ut + 4 * lk + r]);
            const uint16_t *w = P + kW1 + unit * kIn + 16 * lk;
#pragma unroll
            for (int k = 0; k < 16; k += 4) {
                const uint2 wq = load_param4(w + k);
                const f32x4 b = *reinterpret_cast<const f32x4 *>(&T.x[smp][16 * lk + k]);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(wq.x << 16), b[0], acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(wq.x & 0xFFFF0000u), b[1], acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(wq.y << 16), b[2], acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(wq.y & 0xFFFF0000u), b[3], acc, 0, 0, 0);
            }
            f32x4 o;
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] = smp < ns ? fmaxf(acc[r], 0.0f) : 0.0f;
            *reinterpret_cast<f32x4 *>(&T.h1[smp][16 * ut + 4 * lk]) = o;
        }
        __syncthreads();
        // layer 2: inputs 32 lk + k, k = 0..31
        {
            f32x4 acc;
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[r] = bf16_to_f32(P[kB2 + 16 * ut + 4 * lk + r]);
#pragma unroll
            for (int k = 0; k < 32; k += 4) {
                const uint2 wq = *reinterpret_cast<const uint2 *>(&T.w2[unit][32 * lk + k]);
                const f32x4 b = *reinterpret_cast<const f32x4 *>(&T.h1[smp][32 * lk + k]);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(wq.x << 16), b[0], acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(wq.x & 0xFFFF0000u), b[1], acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(wq.y << 16), b[2], acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(wq.y & 0xFFFF0000u), b[3], acc, 0, 0, 0);
            }
            f32x4 o;
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] = smp < ns ? fmaxf(acc[r], 0.0f) : 0.0f;
            *reinterpret_cast<f32x4 *>(&T.h2[smp][16 * ut + 4 * lk]) = o;
        }
        __syncthreads();
        // logits: 32 consecutive lanes per sample, 4 terms each, then a fixed butterfly
        {
            const int s = t >> 5, q = t & 31;
            float acc = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) acc = fmaf(T.h2[s][4 * q + i], bf16_to_f32(P[kW3 + 4 * q + i]), acc);
            for (int o = 1; o < 32; o <<= 1) acc += __shfl_xor(acc, o);
            if (q == 0) T.z[s] = acc + bf16_to_f32(P[kB3]);
        }
        __syncthreads();
        if (t < kTile) {
            float g = 0.0f;
            if (t < ns) {
                const float zz = T.z[t], y = Y[t0 + t], w = WT[t0 + t] * inv_wsum;
                const float p = 1.0f / (1.0f + expf(-zz));
                g = w * (p - y);
                // softplus(z) - y z, in a form that does not overflow
                lsum += w * (fmaxf(zz, 0.0f) + log1pf(expf(-fabsf(zz))) - y * zz);
            }
            T.dz[t] = g;
            gb3 += g;
        }
        __syncthreads();
        // the error at layer 2 (ReLU mask)
        for (int e = t; e < kTile * kH; e += kGradThreads) {
            const int s = e / kH, j = e % kH;
            T.d2[s][j] = T.h2[s][j] > 0.0f ? T.dz[s] * bf16_to_f32(P[kW3 + j]) : 0.0f;
        }
        __syncthreads();
        // layer 3's gradient and layer 2's bias before h2 is overwritten
        if (t < kH) {
#pragma unroll 8
            for (int s = 0; s < kTile; ++s) gsum = fmaf(T.dz[s], T.h2[s][t], gsum);
        } else if (t < 2 * kH) {
#pragma unroll 8
            for (int s = 0; s < kTile; ++s) gsum += T.d2[s][t - kH];
        }
        // error at layer 1: sum_jj d2[s][jj] W2[jj][j] (units 4 k + lk), masked by h1 > 0
        f32x4 e1 = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
        for (int k = 0; k < kH / 4; ++k)
            e1 = __builtin_amdgcn_mfma_f32_16x16x4f32(bf16_to_f32(T.w2[4 * k + lk][unit]), T.d2[smp][4 * k + lk], e1, 0, 0, 0);
        {
            const f32x4 hh = *reinterpret_cast<const f32x4 *>(&T.h1[smp][16 * ut + 4 * lk]);
#pragma unroll
            for (int r = 0; r < 4; ++r) e1[r] = hh[r] > 0.0f ? e1[r] : 0.0f;
        }
        __syncthreads();  // gw3 has read h2
        *reinterpret_cast<f32x4 *>(&T.h2[smp][16 * ut + 4 * lk]) = e1;
        // dW2[r][c] += sum_s d2[s][r] h1[s][c]
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int r0 = 16 * ((4 * wv + q) >> 3), c0 = 16 * ((4 * wv + q) & 7);
#pragma unroll
            for (int k = 0; k < kTile / 4; ++k)
                g2[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(T.d2[4 * k + lk][r0 + li], T.h1[4 * k + lk][c0 + li], g2[q], 0, 0, 0);
        }
        __syncthreads();  // the layer-1 errors are complete
        // dW1[r][c] += sum_s d1[s][r] x[s][c]
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int r0 = 16 * ((2 * wv + q) >> 2), c0 = 16 * ((2 * wv + q) & 3);
#pragma unroll
            for (int k = 0; k < kTile / 4; ++k)
                g1[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(T.h2[4 * k + lk][r0 + li], T.x[4 * k + lk][c0 + li], g1[q], 0, 0, 0);
        }
        if (t >= 2 * kH && t < 3 * kH) {
#pragma unroll 8
            for (int s = 0; s < kTile; ++s) gsum += T.h2[s][t - 2 * kH];
        }
        __syncthreads();  // the next tile overwrites the tile buffers
    }
    float *row = part + (size_t) blockIdx.x * (kMlpParams + 1);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int r0 = 16 * ((4 * wv + q) >> 3), c0 = 16 * ((4 * wv + q) & 7);
#pragma unroll
        for (int r = 0; r < 4; ++r) row[kW2 + (r0 + 4 * lk + r) * kH + c0 + li] = g2[q][r];
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int r0 = 16 * ((2 * wv + q) >> 2), c0 = 16 * ((2 * wv + q) & 3);
#pragma unroll
        for (int r = 0; r < 4; ++r) row[kW1 + (r0 + 4 * lk + r) * kIn + c0 + li] = g1[q][r];
    }
    if (t < kH)
        row[kW3 + t] = gsum;
    else if (t < 2 * kH)
        row[kB2 + t - kH] = gsum;
    else if (t < 3 * kH)
        row[kB1 + t - 2 * kH] = gsum;
    // b3 and the loss: lanes 0..31 hold one sample slot each
    float a = gb3, lo = lsum;
    for (int o = 16; o > 0; o >>= 1) {
        a += __shfl_down(a, o);
        lo += __shfl_down(lo, o);
    }
    if (t == 0) {
        row[kB3] = a;
        row[kMlpParams] = lo;
    }
}

// grad[i] = sum over blocks b of part[b][i], i <= kMlpParams: 64 columns per
// block, four threads per column, each a quarter of the rows in order (16 loads
// in flight), the quarters added in order.  128 rows: 4.7 us; 30 us with one thread per
// column.
constexpr int kRedCols = 64, kRedParts = 4;
__global__ __launch_bounds__(kRedCols * kRedParts) void k_mlp_reduce(const float *__restrict__ part, int nb,
                                                                     float *__restrict__ grad) {
    __shared__ float q[kRedParts][kRedCols];
    const int c = threadIdx.x % kRedCols, g = threadIdx.x / kRedCols;
    const int i = blockIdx.x * kRedCols + c;
    const int per = (nb + kRedParts - 1) / kRedParts, b0 = g * per, b1 = min(nb, b0 + per);
    float s = 0.0f;
    if (i <= kMlpParams) {
        const float *p = part + i;
        int b = b0;
        for (; b + 16 <= b1; b += 16) {
            float v[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) v[u] = p[(size_t) (b + u) * (kMlpParams + 1)];
#pragma unroll
            for (int u = 0; u < 16; ++u) s += v[u];
        }
        for (; b < b1; ++b) s += p[(size_t) b * (kMlpParams + 1)];
    }
    q[g][c] = s;
    __syncthreads();
    if (g == 0 && i <= kMlpParams) grad[i] = (q[0][c] + q[1][c]) + (q[2][c] + q[3][c]);
}

__global__ void k_mlp_adam(float *__restrict__ master, const float *__restrict__ grad, float *__restrict__ m,
                           float *__restrict__ v, uint16_t *__restrict__ P, int n, float lr, float b1, float b2,
                           float c1, float c2, float eps) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float g = grad[i];
    const float mi = b1 * m[i] + (1.0f - b1) * g;
    const float vi = b2 * v[i] + (1.0f - b2) * (g * g);
    m[i] = mi;
    v[i] = vi;
    const float w = master[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    master[i] = w;
    P[i] = f32_to_bf16(w);
}

__global__ void k_mlp_round(const float *__restrict__ master, uint16_t *__restrict__ P, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) P[i] = f32_to_bf16(master[i]);
}

unsigned param_blocks() { return (unsigned) ((kMlpParams + 1 + 255) / 256); }

}  // namespace

hipError_t launch_mlp_round(const float *master, uint16_t *P, hipStream_t st) {
    hipLaunchKernelGGL(k_mlp_round, dim3(param_blocks()), dim3(256), 0, st, master, P, kMlpParams);
    return hipGetLastError();
}

hipError_t launch_mlp_predict(const float *X, long long N, const uint16_t *P, float *prob, hipStream_t st) {
    if (N <= 0) return hipSuccess;
    // four tiles of 32 samples per block at a time; two blocks fill a CU (200,003
    // rows, alone: 41 to 43 us with 512 blocks, 51 with 768 and 54 with 256)
    const long long blocks = (N + 4 * 32 - 1) / (4 * 32);
    const unsigned grid = (unsigned) std::min<long long>(blocks, 2 * 256);
    hipLaunchKernelGGL(k_mlp_predict, dim3(grid), dim3(kThreads), 0, st, X, N, P, prob);
    return hipGetLastError();
}

hipError_t launch_mlp_grad(const float *X, const float *Y, const float *WT, long long N, float inv_wsum,
                           const uint16_t *P, float *part, int nblocks, float *grad, hipStream_t st) {
    if (N <= 0 || nblocks <= 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_mlp_grad, dim3(nblocks), dim3(kGradThreads), 0, st, X, Y, WT, N, inv_wsum, P, part);
    hipLaunchKernelGGL(k_mlp_reduce, dim3((kMlpParams + kRedCols) / kRedCols), dim3(kRedCols * kRedParts), 0, st, part,
                       nblocks, grad);
    return hipGetLastError();
}

hipError_t launch_mlp_adam(float *master, const float *grad, float *m, float *v, uint16_t *P, int step, float lr,
                           hipStream_t st) {
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float c1 = 1.0f - std::pow(b1, (float) step), c2 = 1.0f - std::pow(b2, (float) step);
    hipLaunchKernelGGL(k_mlp_adam, dim3(param_blocks()), dim3(256), 0, st, master, grad, m, v, P, kMlpParams, lr,
                       b1, b2, c1, c2, eps);
    return hipGetLastError();
}

}  // namespace inscy
