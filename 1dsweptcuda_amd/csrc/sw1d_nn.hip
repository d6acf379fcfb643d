// Learned KS surrogate: a periodic 1D convolutional network advancing the KS
// field by K steps at a time, trained and run on gfx950.
//
// Network (6 layers, kernel 5, periodic padding, GELU between layers):
//   L1   1 -> 64 channels   FP32 VALU (5 MACs per output)
//   L2-5 64 -> 64 channels  BF16 MFMA v_mfma_f32_16x16x32_bf16, FP32 accumulate
//   L6   64 -> 1 channel    FP32 VALU over BF16 activations
// output du = L6(...); the integrator adds it to u (residual form).
//
// Activations are channel-last [B][X][64] BF16.  A 64->64 layer is a GEMM per
// tile of 256 (or 64) positions: M = positions, N = output channels, K = 5 taps
// x 64 input channels, staged in LDS in the operand layouts of the MFMA (8
// consecutive K values per lane, 16-byte LDS reads).
//
// Training (one gradient at batch 64 x 1024: 147 us on the GPU, 480 us before)
// keeps two more forms of what a layer computes.  The FP32
// pre-activations Z, for the GELU derivative, are stored in the accumulators'
// own lane order, since only the lanes that hold the same outputs in the
// backward pass read them (16 bytes per lane, no gaps).  And the layer inputs
// and the gradients dZ are stored position-contiguous, [B][64][X], as the
// accumulators hold them (a lane has four positions of one channel): the weight
// gradient is a GEMM over positions (K = positions), whose operands are then
// plain 16-byte loads.  Each workgroup adds its positions' share in registers
// and LDS and writes one partial sum; a second kernel adds the partials in a
// fixed order, so gradients are deterministic.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <type_traits>
#include <utility>
#include <vector>

#include "../../include/swept1d.h"
#include "sw1d_host.hpp"

namespace sw1dnn {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2u __attribute__((ext_vector_type(2), aligned(4)));
typedef __bf16 bf16x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int C = 64;       // hidden channels
constexpr int TAPS = 5;     // kernel width
constexpr int TILE = 64;    // positions nx is a multiple of
constexpr int NT = 256;     // threads per workgroup

// ---------------------------------------------------------------- bf16 ---
// Round to nearest even (NaN kept quiet), the same rule the host oracle uses.
__host__ __device__ inline uint16_t f2bf_bits(float f)
{
    uint32_t u;
    memcpy(&u, &f, 4);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__host__ __device__ inline float bf_bits2f(uint16_t h)
{
    const uint32_t u = (uint32_t)h << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}
// Device rounding uses the hardware conversion (v_cvt_pk_bf16_f32, round to
// nearest even); the device check compares it with f2bf_bits on ties and
// neighbours of ties.
__device__ inline __bf16 f2bf(float f) { return static_cast<__bf16>(f); }
__device__ inline float bf2f(__bf16 h) { return bf_bits2f(__builtin_bit_cast(uint16_t, h)); }

// GELU in its tanh form (Hendrycks & Gimpel; PyTorch's approximate="tanh"):
//   gelu(z) = z sigmoid(c (z + a z^3)),  c = 2 sqrt(2/pi), a = 0.044715,
// i.e. z / (1 + 2^(z (K0 + KA z^2))) with K0 = -c log2(e), KA = a K0: three
// FP32 operations, 2^x and a reciprocal.  Large |z| give z or -0 (2^x goes to
// 0 or inf), never NaN.  Its derivative is s + z s (1 - s) c (1 + 3a z^2),
// s = sigmoid(c (z + a z^3)).
constexpr float GELU_K0 = -2.3022082f;   // -c log2(e)
constexpr float GELU_KA = -0.10294324f;  // a K0
constexpr float GELU_C = 1.5957691f;     // c
constexpr float GELU_C3A = 0.21406445f;  // 3 a c

__device__ inline float gelu_sigmoid(float z)
{
    return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z * fmaf(GELU_KA, z * z, GELU_K0)));
}
__device__ inline float gelu(float z) { return z * gelu_sigmoid(z); }
__device__ inline float gelu_d(float z)
{
    const float s = gelu_sigmoid(z);
    return fmaf(z * s * (1.0f - s), fmaf(GELU_C3A, z * z, GELU_C), s);
}

__device__ inline int wrapx(int x, int X) { return x < 0 ? x + X : (x >= X ? x - X : x); }

// ------------------------------------------------------ MFMA layout check ---
// Assumed v_mfma_f32_16x16x32_bf16 operand layout (lane l = 0..63):
//   A (16x32): lane holds A[l%16][8*(l/16) + j], j = 0..7
//   B (32x16): lane holds B[8*(l/16) + j][l%16]
//   D (16x16): lane holds D[4*(l/16) + j][l%16], j = 0..3
// Checked against a plain product of small integers (exact in BF16/FP32).
__global__ void k_mfma_check(int* ok)
{
    const int l = threadIdx.x;
    bf16x8 a, b;
    for (int j = 0; j < 8; ++j) {
        const int k = 8 * (l / 16) + j;
        a[j] = f2bf((float)(((l % 16) * 3 + k * 5) % 7 - 3));
        b[j] = f2bf((float)((k * 2 + (l % 16) * 7) % 5 - 2));
    }
    f32x4 d = {0.f, 0.f, 0.f, 0.f};
    d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, d, 0, 0, 0);
    for (int j = 0; j < 4; ++j) {
        const int m = 4 * (l / 16) + j, n = l % 16;
        float want = 0.f;
        for (int k = 0; k < 32; ++k)
            want += (float)((m * 3 + k * 5) % 7 - 3) * (float)((k * 2 + n * 7) % 5 - 2);
        if (d[j] != want) atomicAnd(ok, 0);
    }
    // hardware BF16 rounding against the software rule: ties (low half 0x8000)
    // with even and odd kept bits, and their neighbours, over many exponents
    const uint32_t lows[6] = {0x0000u, 0x0001u, 0x7fffu, 0x8000u, 0x8001u, 0xffffu};
    for (int k = 0; k < 6; ++k) {
        const uint32_t bits = ((uint32_t)(l & 1) << 31) | ((uint32_t)(64 + 2 * l) << 23) |
                              ((uint32_t)(l * 37 % 128) << 16) | lows[k];
        float f;
        memcpy(&f, &bits, 4);
        if (__builtin_bit_cast(uint16_t, f2bf(f)) != f2bf_bits(f)) atomicAnd(ok, 0);
    }
}

// ----------------------------------------------- L2-L5: 64 -> 64, MFMA ---
// Z[b][x][co] = bias[co] + sum_t sum_ci A[b][x+t-2][ci] W[t][co][ci]
// over TF positions per workgroup of TF/32 waves, 32 positions x 64 channels
// each (8 accumulator tiles, so four waves fit per SIMD and one workgroup's
// MFMAs overlap another's GELU epilogue).  TF = 256, for the 40 KB of staged
// weights to serve many positions, where nx allows; else 64.
constexpr int TILE_F = 256;
constexpr int WROWS = 32;       // positions per wave
constexpr int MB = WROWS / 16;  // 16-row MFMA blocks per wave
template <int TF> struct Tile {
    static constexpr int NW = TF / WROWS, NT = NW * 64;
};
// Transposed activations [B][64][XT]: position p of a sample at p + 2 of a row
// of XT = X + 8, which also holds the periodic neighbours -2, -1, X, X + 1, so
// that the 12 positions around an 8-position operand start 16-byte aligned.
__host__ __device__ inline int xt(int X) { return X + 8; }

// LDS rows of 64 BF16 (8 chunks of 16 bytes) with chunk c of row r stored at
// chunk c ^ (r & 7): the 16 rows read together by a fragment load hit 8
// different chunk slots, so no padding is needed (2 workgroups fit per CU).
__device__ __forceinline__ int swz(int r, int chunk) { return r * C + ((chunk ^ (r & 7)) << 3); }

// 16-byte chunks of rows of 64 BF16 on their way from memory to an LDS tile:
// every load of a thread is in flight before the first store (one by one they
// cost a memory latency each, 3 us of a 10 us layer).
template <int TF, int ROWS>
struct Staged {
    static constexpr int NT = Tile<TF>::NT, CHUNKS = ROWS * (C / 8), N = (CHUNKS + NT - 1) / NT;
    u32x4 v[N];
    // row r from src(r)
    template <typename F>
    __device__ __forceinline__ void load(F&& src)
    {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int q = threadIdx.x + i * NT;
            if (CHUNKS % NT == 0 || q < CHUNKS)
                v[i] = *reinterpret_cast<const u32x4*>(src(q / (C / 8)) + q % (C / 8) * 8);
        }
    }
    __device__ __forceinline__ void store(__bf16* lds) const
    {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int q = threadIdx.x + i * NT;
            if (CHUNKS % NT == 0 || q < CHUNKS) *reinterpret_cast<u32x4*>(&lds[swz(q / (C / 8), q % (C / 8))]) = v[i];
        }
    }
};
// rows x0-2 .. x0+TF+1 of one sample's [X][64] BF16 activation -> sA, and a
// layer's packed weights [t][co][ci] -> sW (rows t*64 + co)
template <int TF>
__device__ __forceinline__ void stage(__bf16* sA, const __bf16* __restrict__ Ab, int x0, int X, __bf16* sW,
                                      const __bf16* __restrict__ W)
{
    Staged<TF, TF + 4> act;
    Staged<TF, TAPS * C> wts;
    act.load([&](int r) { return Ab + (int64_t)wrapx(x0 - 2 + r, X) * C; });
    wts.load([&](int r) { return W + r * C; });
    act.store(sA);
    wts.store(sW);
}
// Layer 1 evaluated straight into sA: rows x0-2 .. x0+TF+1 of
// bf16(gelu(b1 + sum_t w1[c][t] in[x+t-2])), with in = FP32(u) * inv_scale.
template <int TF, typename TIN>
__device__ __forceinline__ void stage_l1(__bf16* sA, float* sIn, const TIN* __restrict__ ub, float inv_scale,
                                         const float* __restrict__ w1, const float* __restrict__ b1, int x0,
                                         int X)
{
    constexpr int NTW = Tile<TF>::NT;
    for (int q = threadIdx.x; q < TF + 8; q += NTW) sIn[q] = (float)ub[wrapx(x0 - 4 + q, X)] * inv_scale;
    const int c8 = threadIdx.x % (C / 8);  // fixed per thread: NTW is a multiple of 8
    float w[8][TAPS], bb[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        bb[k] = b1[c8 * 8 + k];
#pragma unroll
        for (int t = 0; t < TAPS; ++t) w[k][t] = w1[(c8 * 8 + k) * TAPS + t];
    }
    __syncthreads();
    for (int r = threadIdx.x / (C / 8); r < TF + 4; r += NTW / (C / 8)) {
        bf16x8 v;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            float z = bb[k];
#pragma unroll
            for (int t = 0; t < TAPS; ++t) z = fmaf(w[k][t], sIn[r + t], z);
            v[k] = f2bf(gelu(z));
        }
        *reinterpret_cast<bf16x8*>(&sA[swz(r, c8)]) = v;
    }
}
// acc[mb][nb] = the wave's WROWS positions x 64 channels of
//   FORWARD: sum_t A(x+t-2) W[t]^T;  else: sum_t dZ(x-t+2) W[t]
template <bool FORWARD>
__device__ __forceinline__ void mfma_tile(const __bf16* sA, const __bf16* sW, f32x4 (&acc)[MB][4])
{
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int m0 = WROWS * w, li = l % 16, lq = l / 16;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) acc[mb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
    for (int s = 0; s < TAPS * 2; ++s) {
        const int t = s >> 1, chunk = (s & 1) * 4 + lq;  // K = channels (s&1)*32 + 8*lq ..
        const int row = m0 + li + (FORWARD ? t : 4 - t);
        bf16x8 a[MB], bv[4];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) a[mb] = *reinterpret_cast<const bf16x8*>(&sA[swz(row + 16 * mb, chunk)]);
#pragma unroll
        for (int nb = 0; nb < 4; ++nb)
            bv[nb] = *reinterpret_cast<const bf16x8*>(&sW[swz(t * C + 16 * nb + li, chunk)]);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int nb = 0; nb < 4; ++nb)
                acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[mb], bv[nb], acc[mb][nb], 0, 0, 0);
    }
}
// Z in the accumulators' order: tile, wave, (mb, nb), lane
__device__ __forceinline__ int64_t z_index(int64_t tile, int waves, int w, int mb, int nb, int l)
{
    return (((tile * waves + w) * MB + mb) * 4 + nb) * 64 + l;
}
// four positions x .. x+3 of channel c -> a transposed activation (16 bytes
// would need the neighbour lane's four), and their periodic copies
__device__ __forceinline__ void store_t(__bf16* __restrict__ T, int b, int c, int x, int X, const bf16x4& v)
{
    __bf16* row = T + ((int64_t)b * C + c) * xt(X);
    *reinterpret_cast<bf16x4u*>(row + 2 + x) = v;
    if (x == 0) *reinterpret_cast<bf16x2u*>(row + 2 + X) = bf16x2u{v[0], v[1]};
    if (x == X - 4) *reinterpret_cast<bf16x2u*>(row) = bf16x2u{v[2], v[3]};
}
// bias + GELU of the accumulators, rounded to BF16 into the LDS tile sO (row =
// position in the tile, swizzled).  TRAIN: also the pre-activations to Z (own
// order) and, where T is given, the activations transposed.  sO may alias sA
// once every wave has finished mfma_tile.
template <int TF, bool TRAIN>
__device__ __forceinline__ void epilogue(const f32x4 (&acc)[MB][4], const float* __restrict__ bias, __bf16* sO,
                                         f32x4* __restrict__ Z, __bf16* __restrict__ T, int b, int x0, int X)
{
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int m0 = WROWS * w, li = l % 16, lq = l / 16;
    const int64_t tile = (int64_t)b * (X / TF) + x0 / TF;
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
        const int co = 16 * nb + li;
        const float bc = bias[co];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            const int r = m0 + 16 * mb + 4 * lq;
            f32x4 z;
            bf16x4 a;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                z[j] = acc[mb][nb][j] + bc;
                a[j] = f2bf(gelu(z[j]));
                sO[swz(r + j, co >> 3) + (co & 7)] = a[j];
            }
            if (TRAIN) {
                Z[z_index(tile, Tile<TF>::NW, w, mb, nb, l)] = z;
                if (T) store_t(T, b, co, x0 + r, X, a);
            }
        }
    }
}
// the LDS tile -> rows x0 .. x0+TF-1 of a [X][64] activation (16-byte stores)
template <int TF>
__device__ __forceinline__ void store_act(const __bf16* sO, __bf16* __restrict__ Ab, int x0)
{
    for (int q = threadIdx.x; q < TF * (C / 8); q += Tile<TF>::NT) {
        const int r = q / (C / 8), c8 = q % (C / 8);
        *reinterpret_cast<uint4*>(&Ab[(int64_t)(x0 + r) * C + c8 * 8]) =
            *reinterpret_cast<const uint4*>(&sO[swz(r, c8)]);
    }
}

// One 64 -> 64 layer over TF positions.  TRAIN keeps what the backward pass
// needs (epilogue).
template <int TF, bool TRAIN>
__global__ __launch_bounds__(Tile<TF>::NT) void k_mid_fwd(const __bf16* __restrict__ Ain,
                                                         const __bf16* __restrict__ Wf,
                                                         const float* __restrict__ bias, f32x4* __restrict__ Z,
                                                         __bf16* __restrict__ T, __bf16* __restrict__ Aout, int X)
{
    __shared__ __attribute__((aligned(16))) __bf16 sA[(TF + 4) * C];
    __shared__ __attribute__((aligned(16))) __bf16 sW[TAPS * C * C];
    const int b = blockIdx.y, x0 = blockIdx.x * TF;
    stage<TF>(sA, Ain + (int64_t)b * X * C, x0, X, sW, Wf);
    __syncthreads();
    f32x4 acc[MB][4];
    mfma_tile<true>(sA, sW, acc);
    __syncthreads();
    epilogue<TF, TRAIN>(acc, bias, sA, Z, T, b, x0, X);
    __syncthreads();
    store_act<TF>(sA, Aout + (int64_t)b * X * C, x0);
}

// Layers 1 and 2 in one pass: layer 1 is evaluated into the LDS tile from the
// network input, so its activation goes to memory only where the backward pass
// wants it (TRAIN: transposed, to T1) and its pre-activation never does (the
// backward pass evaluates its five terms again).
template <int TF, typename TIN, bool TRAIN>
__global__ __launch_bounds__(Tile<TF>::NT) void k_l12_fwd(const TIN* __restrict__ in, float inv_scale,
                                                         const float* __restrict__ w1,
                                                         const float* __restrict__ b1,
                                                         const __bf16* __restrict__ Wf,
                                                         const float* __restrict__ bias, __bf16* __restrict__ T1,
                                                         f32x4* __restrict__ Z, __bf16* __restrict__ T,
                                                         __bf16* __restrict__ Aout, int X)
{
    __shared__ __attribute__((aligned(16))) __bf16 sA[(TF + 4) * C];
    __shared__ __attribute__((aligned(16))) __bf16 sW[TAPS * C * C];
    __shared__ float sIn[TF + 8];
    const int b = blockIdx.y, x0 = blockIdx.x * TF;
    Staged<TF, TAPS * C> wts;
    wts.load([&](int r) { return Wf + r * C; });  // in flight during layer 1
    stage_l1<TF, TIN>(sA, sIn, in + (int64_t)b * X, inv_scale, w1, b1, x0, X);
    wts.store(sW);
    __syncthreads();
    if (TRAIN) {
#pragma unroll
        for (int i = 0; i < TF / 4 * C / Tile<TF>::NT; ++i) {
            // a wave: 16 channels x 16 positions (32 contiguous bytes per channel)
            const int q = threadIdx.x + i * Tile<TF>::NT, k = q / 64;
            const int c = 16 * (k % 4) + (q % 64) / 4, r = 16 * (k / 4) + 4 * (q % 4);
            bf16x4 v;
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = sA[swz(r + 2 + j, c >> 3) + (c & 7)];
            store_t(T1, b, c, x0 + r, X, v);
        }
    }
    f32x4 acc[MB][4];
    mfma_tile<true>(sA, sW, acc);
    __syncthreads();
    epilogue<TF, TRAIN>(acc, bias, sA, Z, T, b, x0, X);
    __syncthreads();
    store_act<TF>(sA, Aout + (int64_t)b * X * C, x0);
}

// Layer 5 and the output layer (inference): the BF16 layer-5 tile stays in
// LDS and each thread forms, for its position x, the five tap sums
//   S[t][b*X + x] = sum_c w6[t][c] A5[x][c],
// from which du[x] = b6 + sum_t S[t][x+t-2] (k_l6_out).
constexpr int NTW = Tile<TILE_F>::NT;
static_assert(NTW >= TILE_F, "the output-layer epilogue maps one thread to one position");
__global__ __launch_bounds__(NTW) void k_l56_fwd(const __bf16* __restrict__ Ain, const __bf16* __restrict__ Wf,
                                                const float* __restrict__ bias, const float* __restrict__ w6,
                                                float* __restrict__ S, int X, int64_t plane)
{
    __shared__ __attribute__((aligned(16))) __bf16 sA[(TILE_F + 4) * C];
    __shared__ __attribute__((aligned(16))) __bf16 sW[TAPS * C * C];
    __shared__ float sW6[TAPS * C];
    const int b = blockIdx.y, x0 = blockIdx.x * TILE_F;
    stage<TILE_F>(sA, Ain + (int64_t)b * X * C, x0, X, sW, Wf);
    for (int q = threadIdx.x; q < TAPS * C; q += NTW) sW6[q] = w6[q];
    __syncthreads();
    f32x4 acc[MB][4];
    mfma_tile<true>(sA, sW, acc);
    __syncthreads();
    epilogue<TILE_F, false>(acc, bias, sA, nullptr, nullptr, b, x0, X);
    __syncthreads();
    const int r = threadIdx.x;
    if (r >= TILE_F) return;
    float sum[TAPS] = {0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c8 = 0; c8 < C / 8; ++c8) {
        const bf16x8 v = *reinterpret_cast<const bf16x8*>(&sA[swz(r, c8)]);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float a = bf2f(v[k]);
#pragma unroll
            for (int t = 0; t < TAPS; ++t) sum[t] = fmaf(sW6[t * C + c8 * 8 + k], a, sum[t]);
        }
    }
    const int64_t o = (int64_t)b * X + x0 + r;
#pragma unroll
    for (int t = 0; t < TAPS; ++t) S[t * plane + o] = sum[t];
}

// du = b6 + sum_t S[t][x+t-2] (periodic per sample); APPLY adds out_scale * du
// to the FP64 state in place of storing du (the operation of k_apply_du).
template <bool APPLY>
__global__ __launch_bounds__(NT) void k_l6_out(const float* __restrict__ S, const float* __restrict__ b6,
                                               float* __restrict__ du, const double* u, double* out,
                                               double out_scale, int X, int64_t plane)
{
    const int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x;
    if (i >= plane) return;
    const int x = (int)(i % X);
    const int64_t row = i - x;
    float s = b6[0];
#pragma unroll
    for (int t = 0; t < TAPS; ++t) s += S[t * plane + row + wrapx(x + t - 2, X)];
    if (APPLY)
        out[i] = u[i] + out_scale * (double)s;
    else
        du[i] = s;
}

// parameter vector (FP32), in this order
constexpr int64_t P_W1 = 0, P_B1 = P_W1 + C * TAPS;
constexpr int64_t P_MID = P_B1 + C;                  // 4 x (W[t][co][ci], b[co])
constexpr int64_t MID_SZ = TAPS * C * C + C;
constexpr int64_t P_W6 = P_MID + 4 * MID_SZ, P_B6 = P_W6 + TAPS * C;
constexpr int64_t NPARAM = P_B6 + 1;

// -------------------------------------- whole network, a segment of a sample ---
// Inference at multiples of 256 positions: a workgroup takes SEG positions of a
// periodic sample through all six layers in one launch, its activation (BF16
// rows of 64 channels) in LDS, so no activation goes to memory.
// Tile row q is position p0 - 10 + q: the ten positions on each side that the
// five 5-tap layers reach are the neighbouring segment's, computed here too
// (every layer computes rows 2 .. SEG+17, of which its own reach is exact).
// Each wave owns PB 16-row MFMA blocks, and four waves each take 16 channels of
// the one block left over.  Every value goes through the operations of the
// per-layer kernels in the same order (L1 as stage_l1, the MFMA steps s = 0..9
// of mfma_tile, the epilogue, the tap sums of k_l56_fwd and the sum of
// k_l6_out), so the results are the same bits.
//
// A full chip is bound by issue: 22 us of GELUs (42 cycles per wave and value,
// half of them the exponential and the reciprocal) and 18 us of MFMAs, which
// overlap only in part, also between workgroups (16 GELUs and 16 MFMAs of
// separate waves take 90% of their sum).  A small batch is bound by a
// workgroup's life, the chain of six layers, and a whole sample per workgroup
// left the other CUs idle.  So the segments get smaller with the batch; 64
// samples of 1024 positions take 23 us and 8 take 18, where a workgroup per
// sample took 58 for any batch up to 256, and 256 take 57.  The weights pass through a ring of
// three steps, the next on its way from memory while one is used; they are the
// MFMA's row operand, so that a lane holds four channels of a position, one
// 8-byte store instead of four of 2.
constexpr int STEPS = 2 * TAPS;          // MFMA steps of a layer: 32 input channels of a tap each
constexpr int SLAB = C * 32;             // weights of a step, [co][32 ci]

// One step's weights on their way from memory to a slab in LDS: row co's four
// 16-byte chunks, swizzled so that 16 rows' reads of a chunk meet no bank twice.
template <int NTS>
struct WeightStep {
    static constexpr int EL = SLAB / NTS;
    typedef __bf16 vec __attribute__((ext_vector_type(EL)));
    vec v;
    __device__ __forceinline__ void load(const __bf16* __restrict__ Wf, int s, int tid)
    {
        const int e = tid * EL, co = e / 32;
        v = *reinterpret_cast<const vec*>(&Wf[((s >> 1) * C + co) * C + (s & 1) * 32 + e % 32]);
    }
    __device__ __forceinline__ void store(__bf16* slab, int tid) const
    {
        const int e = tid * EL, co = e / 32, ch = e / 8 % 4;
        *reinterpret_cast<vec*>(&slab[(co * 4 + (ch ^ (co >> 2 & 3))) * 8 + e % 8]) = v;
    }
};

struct MidWeights { const __bf16* w[4]; };  // packed forward weights of L2-L5

// TIN = double: in = FP64 states (normalised by inv_scale), out = in + out_scale
// * du (another array: a neighbouring segment may still have to read in);
// TIN = float: in = network inputs x, du written to du.
template <typename TIN, int SEG, int PB>
__global__ __launch_bounds__(4 * SEG / PB, 4) void k_net_fwd(const TIN* __restrict__ in, float inv_scale,
                                                          const float* __restrict__ P, MidWeights wf,
                                                          float* __restrict__ du, double* __restrict__ out,
                                                          double out_scale, int X)
{
    constexpr int NW = SEG / (16 * PB), NTS = 64 * NW, ROWS = SEG + 20;
    static_assert(NW >= 4 && NTS >= SEG && 3 * SLAB * 2 >= TAPS * (SEG + 4) * 4);
    __shared__ __attribute__((aligned(16))) __bf16 sA[ROWS * C];
    __shared__ __attribute__((aligned(16))) __bf16 sW[3 * SLAB];  // ring of three steps' weights
    __shared__ __attribute__((aligned(16))) float sB[4 * C];      // biases of layers 2-5
    float* sF = reinterpret_cast<float*>(sW + 2 * SLAB);          // network input (before step 2's weights)
    float* sS = reinterpret_cast<float*>(sW);                     // output-layer tap sums (after layer 5)
    const int tid = threadIdx.x, nseg = X / SEG, p0 = (int)(blockIdx.x % nseg) * SEG;
    const int64_t row = (int64_t)(blockIdx.x / nseg) * X;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    WeightStep<NTS> w0, w1, ws;
    w0.load(wf.w[0], 0, tid);
    w1.load(wf.w[0], 1, tid);
    ws.load(wf.w[0], 2, tid);
    // layer 1 (stage_l1) into every tile row
    for (int i = tid; i < ROWS + 4; i += NTS)
        sF[i] = (float)in[row + wrapx(p0 - 12 + i, X)] * inv_scale;
    if (tid < 4 * C) sB[tid] = P[P_MID + (tid / C) * MID_SZ + TAPS * C * C + tid % C];
    {
        const int c8 = tid % (C / 8);
        float w[8][TAPS], bb[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            bb[k] = P[P_B1 + c8 * 8 + k];
#pragma unroll
            for (int t = 0; t < TAPS; ++t) w[k][t] = P[P_W1 + (c8 * 8 + k) * TAPS + t];
        }
        w0.store(sW, tid);
        w1.store(sW + SLAB, tid);
        __syncthreads();
        for (int q = tid / (C / 8); q < ROWS; q += NTS / (C / 8)) {
            bf16x8 v;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                float z = bb[k];
#pragma unroll
                for (int t = 0; t < TAPS; ++t) z = fmaf(w[k][t], sF[q + t], z);
                v[k] = f2bf(gelu(z));
            }
            *reinterpret_cast<bf16x8*>(&sA[swz(q, c8)]) = v;
        }
    }

    // layers 2-5: acc[cb][pb] is channels 16 cb + 4 lq + j of row 16 (4 wave + pb)
    // + li + 2 (the weights are the MFMA's row operand, so a lane's four values are
    // 8 bytes of the tile)
    const bool extra = wave < 4;
    for (int layer = 0; layer < 4; ++layer) {
        // with 128 registers, addresses recomputed per layer rather than kept
        // live across it
        int lane = tid;
        if constexpr (PB == 4) asm volatile("" : "+v"(lane));
        const int li = lane % 16, lq = lane / 16 % 4, row0 = 16 * PB * wave + li, rowe = 16 * PB * NW + li;
        f32x4 acc[4][PB], acce = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int cb = 0; cb < 4; ++cb)
#pragma unroll
            for (int pb = 0; pb < PB; ++pb) acc[cb][pb] = f32x4{0.f, 0.f, 0.f, 0.f};
        int slot = layer % 3;  // of the layer's step 0: 10 layer mod 3
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            // the input of the layer and this step's weights are complete, and
            // the previous step's are no longer read
            __syncthreads();
            const int free = slot == 0 ? 2 : slot - 1;
            if (s + 2 < STEPS || layer < 3) ws.store(sW + free * SLAB, tid);
            if (s + 3 < STEPS)
                ws.load(wf.w[layer], s + 3, tid);
            else if (layer < 3)
                ws.load(wf.w[layer + 1], s + 3 - STEPS, tid);
            if (s == 0) __builtin_amdgcn_s_setprio(1);
            const __bf16* slab = sW + slot * SLAB;
            slot = slot == 2 ? 0 : slot + 1;

            const int t = s >> 1, chunk = (s & 1) * 4 + lq;
            const __bf16* px = &sA[swz(row0 + t, chunk)];                     // + 16 rows per block
            const __bf16* pw = slab + (li * 4 + (lq ^ (li >> 2 & 3))) * 8;    // + 16 rows per block
            bf16x8 w[4], x[PB];
#pragma unroll
            for (int cb = 0; cb < 4; ++cb) w[cb] = *reinterpret_cast<const bf16x8*>(pw + 16 * 32 * cb);
#pragma unroll
            for (int pb = 0; pb < PB; ++pb) x[pb] = *reinterpret_cast<const bf16x8*>(px + 16 * pb * C);
#pragma unroll
            for (int cb = 0; cb < 4; ++cb)
#pragma unroll
                for (int pb = 0; pb < PB; ++pb)
                    acc[cb][pb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[cb], x[pb], acc[cb][pb], 0, 0, 0);
            if (extra) {
                const bf16x8 we = *reinterpret_cast<const bf16x8*>(pw + 16 * 32 * wave);
                const bf16x8 xe = *reinterpret_cast<const bf16x8*>(&sA[swz(rowe + t, chunk)]);
                acce = __builtin_amdgcn_mfma_f32_16x16x32_bf16(we, xe, acce, 0, 0, 0);
            }
        }
        __builtin_amdgcn_s_setprio(0);
        auto activate = [&](const f32x4& a, int cb) {
            const f32x4 bc = *reinterpret_cast<const f32x4*>(&sB[layer * C + 16 * cb + 4 * lq]);
            bf16x4 o;
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = f2bf(gelu(a[j] + bc[j]));
            return o;
        };
        auto place = [&](int row, int cb, const bf16x4& o) {
            *reinterpret_cast<bf16x4*>(&sA[swz(row + 2, 2 * cb + (lq >> 1)) + 4 * (lq & 1)]) = o;
        };
        bf16x4 o[4][PB], oe;
#pragma unroll
        for (int cb = 0; cb < 4; ++cb)
#pragma unroll
            for (int pb = 0; pb < PB; ++pb) o[cb][pb] = activate(acc[cb][pb], cb);
        if (extra) oe = activate(acce, wave);
        __syncthreads();  // every wave has read the layer input: overwrite it in place
#pragma unroll
        for (int cb = 0; cb < 4; ++cb)
#pragma unroll
            for (int pb = 0; pb < PB; ++pb) place(row0 + 16 * pb, cb, o[cb][pb]);
        if (extra) place(rowe, wave, oe);
    }
    __syncthreads();

    // output layer: the five tap sums S[t][i] of rows 8 + i (k_l56_fwd), i = 0 ..
    // SEG+3, then du = b6 + sum_t S[t][i+t] (k_l6_out).  The weights of a thread's
    // own row are scalar operands; 20 threads add one sum of the four rows beyond.
    const float* __restrict__ w6 = P + P_W6;
    if (tid < SEG) {
        float sum[TAPS] = {0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c8 = 0; c8 < C / 8; ++c8) {
            const bf16x8 v = *reinterpret_cast<const bf16x8*>(&sA[swz(tid + 10, c8)]);
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const float a = bf2f(v[k]);
#pragma unroll
                for (int t = 0; t < TAPS; ++t) sum[t] = fmaf(w6[t * C + c8 * 8 + k], a, sum[t]);
            }
        }
#pragma unroll
        for (int t = 0; t < TAPS; ++t) sS[t * (SEG + 4) + tid + 2] = sum[t];
    }
    if (tid < 4 * TAPS) {
        const int t = tid % TAPS, e = tid / TAPS, i = e < 2 ? e : SEG + e;
        float sum = 0.f;
        for (int c8 = 0; c8 < C / 8; ++c8) {
            const bf16x8 v = *reinterpret_cast<const bf16x8*>(&sA[swz(i + 8, c8)]);
#pragma unroll
            for (int k = 0; k < 8; ++k) sum = fmaf(w6[t * C + c8 * 8 + k], bf2f(v[k]), sum);
        }
        sS[t * (SEG + 4) + i] = sum;
    }
    __syncthreads();
    if (tid >= SEG) return;
    const int64_t o = row + p0 + tid;
    float s = P[P_B6];
#pragma unroll
    for (int t = 0; t < TAPS; ++t) s += sS[t * (SEG + 4) + tid + t];
    if (out)
        out[o] = (double)in[o] + out_scale * (double)s;
    else
        du[o] = s;
}

// ------------------------------------------------------ L6: 64 -> 1, VALU ---
// du[b][x] = b6 + sum_t sum_ci w6[t][ci] A5[b][x+t-2][ci], one thread per
// position.  LOSS: against the target, g = d loss / d du = 2 (du - target) / N
// and the block's sum of (du - target)^2 (loss = their mean over the batch).
template <bool LOSS>
__global__ __launch_bounds__(NT) void k_l6_fwd(const __bf16* __restrict__ A, const float* __restrict__ w6,
                                               const float* __restrict__ b6, float* __restrict__ du,
                                               const float* __restrict__ tgt, float* __restrict__ g,
                                               float* __restrict__ part, int X, int64_t N)
{
    __shared__ float red[NT];
    const int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x;
    float e = 0.f;
    if (i < N) {
        const int x = (int)(i % X);
        const __bf16* Ab = A + (i - x) * C;
        float s = b6[0];
#pragma unroll
        for (int t = 0; t < TAPS; ++t) {
            const bf16x8* row = reinterpret_cast<const bf16x8*>(Ab + (int64_t)wrapx(x + t - 2, X) * C);
#pragma unroll
            for (int c8 = 0; c8 < C / 8; ++c8) {
                const bf16x8 v = row[c8];
#pragma unroll
                for (int k = 0; k < 8; ++k) s = fmaf(w6[t * C + c8 * 8 + k], bf2f(v[k]), s);
            }
        }
        if (LOSS) {
            const float d = s - tgt[i];
            g[i] = 2.f * d / (float)N;
            e = d * d;
        } else {
            du[i] = s;
        }
    }
    if (!LOSS) return;
    red[threadIdx.x] = e;
    __syncthreads();
    for (int s = NT / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// ------------------------------------------------------------- backward ---
// A layer's gradient dZ leaves in two forms: row-major (through the LDS tile
// sD) for the next backward product, and, where T is given, transposed
// ([B][64][X], no neighbours) for the weight gradient.
__device__ __forceinline__ void put_dz(__bf16* sD, __bf16* __restrict__ T, int b, int c, int x0, int r, int X,
                                       const bf16x4& d)
{
#pragma unroll
    for (int j = 0; j < 4; ++j) sD[swz(r + j, c >> 3) + (c & 7)] = d[j];
    if (T) *reinterpret_cast<bf16x4*>(T + ((int64_t)b * C + c) * X + x0 + r) = d;
}

// dA5[b][y][ci] = sum_t g[b][y-t+2] w6[t][ci];  dZ5 = bf16(dA5 * gelu'(Z5)),
// in the lane order of the forward accumulators, which is Z's.
template <int TF>
__global__ __launch_bounds__(Tile<TF>::NT) void k_l6_bwd_data(const float* __restrict__ g,
                                                             const float* __restrict__ w6,
                                                             const f32x4* __restrict__ Z5, __bf16* __restrict__ T,
                                                             __bf16* __restrict__ dZ5, int X)
{
    __shared__ __attribute__((aligned(16))) __bf16 sD[TF * C];
    __shared__ float sG[TF + 4];
    const int b = blockIdx.y, x0 = blockIdx.x * TF;
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6, li = l % 16, lq = l / 16;
    for (int q = threadIdx.x; q < TF + 4; q += Tile<TF>::NT) sG[q] = g[(int64_t)b * X + wrapx(x0 - 2 + q, X)];
    __syncthreads();
    const int64_t tile = (int64_t)b * (X / TF) + blockIdx.x;
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
        const int ci = 16 * nb + li;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            const int r = WROWS * w + 16 * mb + 4 * lq;
            const f32x4 z = Z5[z_index(tile, Tile<TF>::NW, w, mb, nb, l)];
            bf16x4 d;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float s = 0.f;
#pragma unroll
                for (int t = 0; t < TAPS; ++t) s += sG[r + j - t + 4] * w6[t * C + ci];
                d[j] = f2bf(s * gelu_d(z[j]));
            }
            put_dz(sD, T, b, ci, x0, r, X, d);
        }
    }
    __syncthreads();
    store_act<TF>(sD, dZ5 + (int64_t)b * X * C, x0);
}

// dA[b][y][ci] = sum_t sum_co dZ[b][y-t+2][co] W[t][co][ci]   (W as Wb[t][ci][co])
// then dZprev = bf16(dA * gelu'(Zprev)).  FIRST: the previous layer is layer 1,
// whose Z is its five terms of the input again (stage_l1's, in their order).
template <int TF, bool FIRST>
__global__ __launch_bounds__(Tile<TF>::NT) void k_mid_bwd_data(const __bf16* __restrict__ dZ,
                                                              const __bf16* __restrict__ Wb,
                                                              const f32x4* __restrict__ Zprev,
                                                              const float* __restrict__ in,
                                                              const float* __restrict__ w1,
                                                              const float* __restrict__ b1, __bf16* __restrict__ T,
                                                              __bf16* __restrict__ dZprev, int X)
{
    __shared__ __attribute__((aligned(16))) __bf16 sD[(TF + 4) * C];
    __shared__ __attribute__((aligned(16))) __bf16 sW[TAPS * C * C];
    __shared__ float sIn[FIRST ? TF + 4 : 1];
    const int b = blockIdx.y, y0 = blockIdx.x * TF;
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6, li = l % 16, lq = l / 16;
    const int64_t tile = (int64_t)b * (X / TF) + blockIdx.x;
    if (FIRST)
        for (int q = threadIdx.x; q < TF + 4; q += Tile<TF>::NT) sIn[q] = in[(int64_t)b * X + wrapx(y0 - 2 + q, X)];
    stage<TF>(sD, dZ + (int64_t)b * X * C, y0, X, sW, Wb);
    f32x4 z[MB][4];  // in flight during the product
    if (!FIRST) {
#pragma unroll
        for (int nb = 0; nb < 4; ++nb)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) z[mb][nb] = Zprev[z_index(tile, Tile<TF>::NW, w, mb, nb, l)];
    }
    __syncthreads();
    f32x4 acc[MB][4];
    mfma_tile<false>(sD, sW, acc);
    __syncthreads();
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
        const int ci = 16 * nb + li;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            const int r = WROWS * w + 16 * mb + 4 * lq;
            if (FIRST) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float v = b1[ci];
#pragma unroll
                    for (int t = 0; t < TAPS; ++t) v = fmaf(w1[ci * TAPS + t], sIn[r + j + t], v);
                    z[mb][nb][j] = v;
                }
            }
            bf16x4 d;
#pragma unroll
            for (int j = 0; j < 4; ++j) d[j] = f2bf(acc[mb][nb][j] * gelu_d(z[mb][nb][j]));
            put_dz(sD, T, b, ci, y0, r, X, d);
        }
    }
    __syncthreads();
    store_act<TF>(sD, dZprev + (int64_t)b * X * C, y0);
}

// ------------------------------------------------------ weight gradients ---
// One launch for every layer: blockIdx.y = 0 .. 3 the 64 -> 64 layers, 4 the
// output layer, 5 layer 1; blockIdx.x = the share of the positions.  Partial
// sums, one set per share: part[y][x][..] (offsets PART_OFF).
//   64 -> 64: dW[t][co][ci] = sum_x dZ[x][co] A[x+t-2][ci];  db[co] = sum_x dZ[x][co]
// Wave w of 8 takes a 32 x 32 quarter of (co, ci) for every tap and every
// second group of 32 positions: 80 accumulators per lane and two more MFMAs per
// group for db (B = 1).  A lane loads 8 positions of dZ^T and the 12 positions
// -2 .. 9 of A^T around them; the five taps' operands are that window shifted,
// with no LDS.  The two waves of a quarter then add up through LDS (in the
// accumulators' order, which k_reduce_grad undoes).
// At most 256 workgroups of 8 waves, one per CU, so that all run at once: 52 for
// each 64 -> 64 layer and 24 for each edge layer, whose rounds are shorter (64
// for each of the six left a second round of edge workgroups: a training
// iteration of 64 samples 155.7 -> 152.5 us, of 8 103.4 -> 100.1).  17 MB of
// partials for all layers, where one partial per 64 positions was 84 MB per layer.  All
// weight gradients and their reduction: 35 us (67 MB of operands, 13 us at the
// copy rate, then the partials), where a launch per layer with operands
// transposed through LDS and a two-pass reduction took 340 us.
constexpr int MID_SHARES = 52, EDGE_SHARES = 24;
constexpr int WG_SHARES = MID_SHARES;  // partials that the buffer holds for each layer
constexpr int NTG = 512;
constexpr int64_t MIDP = TAPS * C * C + C;    // a 64 -> 64 layer's partial
constexpr int64_t OUTP = TAPS * C + 1;        // the output layer's
constexpr int64_t FIRSTP = C * TAPS + C;      // layer 1's
__host__ __device__ inline int64_t part_offset(int y)
{
    return (y <= 4 ? y * MIDP : 4 * MIDP + OUTP) * WG_SHARES;
}
struct GradIn {
    const __bf16* dzt[4];  // dZ of L2..L5, [B][64][X]
    const __bf16* at[4];   // their inputs A1..A4, [B][64][xt(X)]
    const float* g;        // d loss / d du, [B][X]
    const __bf16* a5;      // [B][X][64]
    const __bf16* dz1;     // [B][X][64]
    const float* in;       // [B][X]
};

__device__ __forceinline__ bf16x8 window_tap(const uint32_t (&d)[6], int t)
{
    uint32_t r[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
        r[k] = t & 1 ? __builtin_amdgcn_alignbit(d[t / 2 + k + 1], d[t / 2 + k], 16) : d[t / 2 + k];
    return __builtin_bit_cast(bf16x8, r);
}

__device__ __forceinline__ void grad_mid(const __bf16* __restrict__ dzt, const __bf16* __restrict__ at,
                                         float* __restrict__ part, float* lds, int X, int groups, int share,
                                         int shares)
{
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6, li = l % 16, lq = l / 16;
    const int qco = w & 1, qci = (w >> 1) & 1, pg = w >> 2;
    const int per = (groups + shares - 1) / shares;
    const int k0 = share * per, k1 = k0 + per < groups ? k0 + per : groups;
    const int gx = X / 32;  // groups of 32 positions per sample
    f32x4 acc[TAPS][2][2], accb[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        accb[m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < TAPS; ++t)
#pragma unroll
            for (int n = 0; n < 2; ++n) acc[t][m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    bf16x8 one;
#pragma unroll
    for (int j = 0; j < 8; ++j) one[j] = f2bf(1.f);
    struct Operands { uint4 a[2]; uint4 b0[2]; uint2 b1[2]; };
    auto load = [&](int k, Operands& o) {
        const int b = k / gx, x = (k % gx) * 32 + 8 * lq;
#pragma unroll
        for (int m = 0; m < 2; ++m)
            o.a[m] = *reinterpret_cast<const uint4*>(dzt + ((int64_t)b * C + 32 * qco + 16 * m + li) * X + x);
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            const __bf16* p = at + ((int64_t)b * C + 32 * qci + 16 * n + li) * xt(X) + x;  // position x - 2
            o.b0[n] = *reinterpret_cast<const uint4*>(p);
            o.b1[n] = *reinterpret_cast<const uint2*>(p + 8);
        }
    };
    auto product = [&](const Operands& o) {
        bf16x8 a[2];
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            a[m] = __builtin_bit_cast(bf16x8, o.a[m]);
            accb[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], one, accb[m], 0, 0, 0);
        }
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            const uint32_t d[6] = {o.b0[n].x, o.b0[n].y, o.b0[n].z, o.b0[n].w, o.b1[n].x, o.b1[n].y};
#pragma unroll
            for (int t = 0; t < TAPS; ++t) {
                const bf16x8 bv = window_tap(d, t);
#pragma unroll
                for (int m = 0; m < 2; ++m)
                    acc[t][m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], bv, acc[t][m][n], 0, 0, 0);
            }
        }
    };
    // two groups' operands are in flight while one multiplies
    Operands o0, o1;
    int k = k0 + pg;
    if (k < k1) load(k, o0);
    if (k + 2 < k1) load(k + 2, o1);
    for (; k < k1; k += 4) {
        product(o0);
        if (k + 4 < k1) load(k + 4, o0);
        if (k + 2 < k1) {
            product(o1);
            if (k + 6 < k1) load(k + 6, o1);
        }
    }
    // [quarter][tap, m, n][lane] float4, then [co] bias sums
    f32x4* sum = reinterpret_cast<f32x4*>(lds) + (w & 3) * (TAPS * 4 * 64) + l;
    f32x4* out = reinterpret_cast<f32x4*>(part) + (w & 3) * (TAPS * 4 * 64) + l;
    float* sb = lds + TAPS * C * C;
    if (pg == 1) {
#pragma unroll
        for (int t = 0; t < TAPS; ++t)
#pragma unroll
            for (int m = 0; m < 2; ++m)
#pragma unroll
                for (int n = 0; n < 2; ++n) sum[((t * 2 + m) * 2 + n) * 64] = acc[t][m][n];
        if (qci == 0 && li == 0) {
#pragma unroll
            for (int m = 0; m < 2; ++m)
                *reinterpret_cast<f32x4*>(sb + 32 * qco + 16 * m + 4 * lq) = accb[m];
        }
    }
    __syncthreads();
    if (pg == 0) {
#pragma unroll
        for (int t = 0; t < TAPS; ++t)
#pragma unroll
            for (int m = 0; m < 2; ++m)
#pragma unroll
                for (int n = 0; n < 2; ++n) {
                    const int f = ((t * 2 + m) * 2 + n) * 64;
                    out[f] = acc[t][m][n] + sum[f];
                }
        if (qci == 0 && li == 0) {
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const int co = 32 * qco + 16 * m + 4 * lq;
                *reinterpret_cast<f32x4*>(part + TAPS * C * C + co) = accb[m] + *reinterpret_cast<f32x4*>(sb + co);
            }
        }
    }
}

// The first and the output layer: rows x of 64 channels (row-major BF16, each
// loaded once, 16 bytes per lane: lane l takes channels 8 (l & 7) .. + 7 of
// every eighth row) against five shifted FP32 values, over segments of 64
// positions, one per wave and round:
//   OUT:   acc[t] += A[x+t-2] g[x]  (A the rows; g outside the segment is 0)
//   else:  acc[t] += dZ[x] in[x+t-2], acc[5] += dZ[x]
template <bool OUT>
__device__ __forceinline__ void grad_edge(const __bf16* __restrict__ rows, const float* __restrict__ f,
                                          float* __restrict__ part, float* lds, int X, int groups, int share,
                                          int shares)
{
    constexpr int ROWS = OUT ? 68 : 64, NR = (ROWS + 7) / 8;
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6, c8 = l & 7, rr = l >> 3;
    const int segs = groups / 2, per = (segs + shares - 1) / shares;
    const int s0 = share * per, s1 = s0 + per < segs ? s0 + per : segs;
    const int sx = X / 64;
    float* sf = lds + w * 80;  // this wave's f[x0 - 4 .. x0 + 67], then zeros
    float acc[TAPS + 1][8];
#pragma unroll
    for (int t = 0; t <= TAPS; ++t)
#pragma unroll
        for (int k = 0; k < 8; ++k) acc[t][k] = 0.f;
    float sum = 0.f;  // OUT: the lane's share of sum g
    // the waves of a workgroup run the same number of rounds (barriers)
    for (int k = 0; k < (per + 7) / 8; ++k) {
        const int s = s0 + k * 8 + w;
        const bool live = s < s1;
        const int b = live ? s / sx : 0, x0 = live ? (s % sx) * 64 : 0;
        const float* fb = f + (int64_t)b * X;
        const __bf16* rb = rows + (int64_t)b * X * C + c8 * 8;
        bf16x8 v[NR];
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int r = i * 8 + rr;
            v[i] = *reinterpret_cast<const bf16x8*>(rb + (int64_t)wrapx(OUT ? x0 - 2 + r : x0 + r, X) * C);
        }
        __syncthreads();
        for (int q = l; q < 80; q += 64) {
            const int x = x0 - 4 + q;
            const bool in = live && q < 72 && (!OUT || (x >= x0 && x < x0 + 64));
            sf[q] = in ? fb[wrapx(x, X)] : 0.f;
        }
        __syncthreads();
        if (!live) continue;
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            // OUT: row x0 - 2 + r meets g[x0 + r - t] (a ninth row past 67 meets
            // zeros only); else row x0 + r meets in[x0 + r + t - 2]
            const int r = i * 8 + rr;
            float e[TAPS];
#pragma unroll
            for (int t = 0; t < TAPS; ++t) e[t] = OUT ? sf[r - t + 4] : sf[r + t + 2];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const float a = bf2f(v[i][q]);
#pragma unroll
                for (int t = 0; t < TAPS; ++t) acc[t][q] = fmaf(e[t], a, acc[t][q]);
                if (!OUT) acc[TAPS][q] += a;
            }
        }
        if (OUT) sum += sf[l + 4];
    }
    __syncthreads();
    // lds: [tap][wave][row lane][channel], then the waves' sums of g
    constexpr int NA = OUT ? TAPS : TAPS + 1;
#pragma unroll
    for (int t = 0; t < NA; ++t)
#pragma unroll
        for (int q = 0; q < 8; ++q) lds[((t * 8 + w) * 8 + rr) * C + c8 * 8 + q] = acc[t][q];
    if (OUT) {
        for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
        if (l == 0) lds[NA * 64 * C + w] = sum;
    }
    __syncthreads();
    for (int q = threadIdx.x; q < NA * C; q += NTG) {
        const int t = q / C, c = q % C;
        float s = 0.f;
#pragma unroll 16
        for (int v = 0; v < 64; ++v) s += lds[(t * 64 + v) * C + c];
        part[OUT ? q : (t < TAPS ? c * TAPS + t : TAPS * C + c)] = s;
    }
    if (OUT && threadIdx.x == 0) {
        float s = 0.f;
        for (int v = 0; v < 8; ++v) s += lds[NA * 64 * C + v];
        part[TAPS * C] = s;
    }
}

__global__ __launch_bounds__(NTG) void k_grad_weights(GradIn in, float* __restrict__ part, int X, int groups,
                                                      int mids, int edges)
{
    // the edge layers' sums, the largest user: 6 taps x 64 lanes of rows x 64 channels
    constexpr int64_t LDS = 6 * 64 * C > MIDP ? 6 * 64 * C : MIDP;
    __shared__ __attribute__((aligned(16))) float lds[LDS];
    const bool mid = (int)blockIdx.x < 4 * mids;
    const int shares = mid ? mids : edges, k = blockIdx.x - (mid ? 0 : 4 * mids);
    const int y = k / shares + (mid ? 0 : 4), share = k % shares;
    float* p = part + part_offset(y) + share * (y < 4 ? MIDP : (y == 4 ? OUTP : FIRSTP));
    if (y < 4)
        grad_mid(in.dzt[y], in.at[y], p, lds, X, groups, share, shares);
    else if (y == 4)
        grad_edge<true>(in.a5, in.g, p, lds, X, groups, share, shares);
    else
        grad_edge<false>(in.dz1, in.in, p, lds, X, groups, share, shares);
}

// g[i] = the sum of the shares' partials in share order, one thread per
// parameter, in the order the partials are stored in.
__global__ __launch_bounds__(NT) void k_reduce_grad(const float* __restrict__ part, int mids, int edges,
                                                    float* __restrict__ g)
{
    int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x;
    if (i >= NPARAM) return;
    int y = 0;
    int64_t len = MIDP, out;
    if (i < 4 * MIDP) {
        y = (int)(i / MIDP);
        i -= y * MIDP;
        out = P_MID + y * MID_SZ;
        if (i < TAPS * C * C) {
            // [quarter][t, m, n][lane][j] -> [t][co][ci]
            const int j = i & 3, l = (i >> 2) & 63, f = (int)(i >> 8);
            const int n = f & 1, m = (f >> 1) & 1, t = (f >> 2) % TAPS, q = f / (4 * TAPS);
            out += (t * C + 32 * (q & 1) + 16 * m + 4 * (l / 16) + j) * C + 32 * (q >> 1) + 16 * n + l % 16;
        } else {
            out += i;
        }
    } else if (i < 4 * MIDP + OUTP) {
        y = 4;
        i -= 4 * MIDP;
        len = OUTP;
        out = P_W6 + i;
    } else {
        y = 5;
        i -= 4 * MIDP + OUTP;
        len = FIRSTP;
        out = P_W1 + i;
    }
    const float* p = part + part_offset(y) + i;
    const int shares = y < 4 ? mids : edges;
    float s = 0.f;
#pragma unroll 8
    for (int k = 0; k < shares; ++k) s += p[k * len];
    g[out] = s;
}

// -------------------------------------------------------------- optimiser ---
__global__ __launch_bounds__(NT) void k_adam(float* __restrict__ p, const float* __restrict__ g,
                                             float* __restrict__ m, float* __restrict__ v, int64_t n,
                                             float lr, float b1, float b2, float eps, float c1, float c2)
{
    const int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// BF16 copies of the 64->64 layers' weights in the forward ([t][co][ci]) and
// backward ([t][ci][co]) layouts, one layer per blockIdx.y.
struct PackOut { __bf16 *wf[4], *wb[4]; };
__global__ __launch_bounds__(NT) void k_pack_w(const float* __restrict__ p, PackOut o)
{
    const int i = blockIdx.x * NT + threadIdx.x;
    if (i >= TAPS * C * C) return;
    const float* w = p + P_MID + blockIdx.y * MID_SZ;
    __bf16 *wf = o.wf[blockIdx.y], *wb = o.wb[blockIdx.y];
    const int t = i / (C * C), co = (i / C) % C, ci = i % C;
    const __bf16 h = f2bf(w[i]);
    wf[i] = h;
    wb[(t * C + ci) * C + co] = h;
}

// out = u + scale * du
__global__ __launch_bounds__(NT) void k_apply_du(const double* u, const float* __restrict__ du, double* out,
                                                 int64_t n, double scale)
{
    const int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x;
    if (i < n) out[i] = u[i] + scale * (double)du[i];
}

// Judged step: u[p] <- unn[p] for the problems whose network state is kept.
__global__ __launch_bounds__(NT) void k_keep_rows(double* __restrict__ u, const double* __restrict__ unn,
                                                  const int* __restrict__ keep, int X, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x;
    if (i < n && keep[i / X]) u[i] = unn[i];
}

// Training mini-batch: row b of (x, t) <- sample idx[b] of the stored set.
__global__ __launch_bounds__(NT) void k_gather(const float* __restrict__ sx, const float* __restrict__ st,
                                               const int64_t* __restrict__ idx, float* __restrict__ x,
                                               float* __restrict__ t, int X, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x;
    if (i >= n) return;
    const int64_t b = i / X, src = idx[b] * X + (i - b * X);
    x[i] = sx[src];
    t[i] = st[src];
}

// Relative L2 distance ||a - b|| / ||b|| partial sums per block: (sum (a-b)^2, sum
// b^2).  Block (k, p) adds points k NT .. of problem p, whose last block may be a
// part of one (X is a multiple of 64).
__global__ __launch_bounds__(NT) void k_l2_parts(const double* __restrict__ a, const double* __restrict__ b, int X,
                                                 double* __restrict__ part)
{
    __shared__ double r0[NT], r1[NT];
    const int x = blockIdx.x * NT + threadIdx.x;
    const int64_t i = (int64_t)blockIdx.y * X + x;
    double d = 0, s = 0;
    if (x < X) {
        d = (a[i] - b[i]) * (a[i] - b[i]);
        s = b[i] * b[i];
    }
    r0[threadIdx.x] = d;
    r1[threadIdx.x] = s;
    __syncthreads();
    for (int k = NT / 2; k > 0; k >>= 1) {
        if (threadIdx.x < k) {
            r0[threadIdx.x] += r0[threadIdx.x + k];
            r1[threadIdx.x] += r1[threadIdx.x + k];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const int64_t k = (int64_t)blockIdx.y * gridDim.x + blockIdx.x;
        part[2 * k] = r0[0];
        part[2 * k + 1] = r1[0];
    }
}

__global__ __launch_bounds__(NT) void k_zero_f64(double* __restrict__ a, int64_t n)
{
    for (int64_t i = threadIdx.x; i < n; i += NT) a[i] = 0.0;
}

// The judge's decision, one block: problem p's relative L2 distance from the
// partial sums of its `per` blocks (added in block order), keep[p] = err <=
// tol (the network's state stays), and over the call acc[0] += the number of
// fallbacks, acc[1] = max(acc[1], largest err).  A NaN distance falls back
// and leaves the maximum unchanged.
__global__ __launch_bounds__(NT) void k_judge(const double* __restrict__ part, int64_t B, int64_t per,
                                              double tol, int* __restrict__ keep, double* __restrict__ acc)
{
    __shared__ double smax[NT], scnt[NT];
    double mx = 0.0, cnt = 0.0;
    for (int64_t p = threadIdx.x; p < B; p += NT) {
        double d = 0, s = 0;
        for (int64_t k = p * per; k < (p + 1) * per; ++k) {
            d += part[2 * k];
            s += part[2 * k + 1];
        }
        const double err = s > 0 ? sqrt(d / s) : sqrt(d);
        mx = err > mx ? err : mx;
        keep[p] = err <= tol;
        cnt += err <= tol ? 0.0 : 1.0;
    }
    smax[threadIdx.x] = mx;
    scnt[threadIdx.x] = cnt;
    __syncthreads();
    for (int k = NT / 2; k > 0; k >>= 1) {
        if (threadIdx.x < k) {
            smax[threadIdx.x] = smax[threadIdx.x + k] > smax[threadIdx.x] ? smax[threadIdx.x + k] : smax[threadIdx.x];
            scnt[threadIdx.x] += scnt[threadIdx.x + k];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        acc[0] += scnt[0];
        acc[1] = smax[0] > acc[1] ? smax[0] : acc[1];
    }
}

}  // namespace sw1dnn

// ================================================================== host ===
namespace sw1dnn {

inline unsigned nblk(int64_t n) { return (unsigned)((n + NT - 1) / NT); }

uint64_t splitmix(uint64_t& s)
{
    uint64_t z = (s += 0x9E3779B97F4A7C15ULL);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}
double normal(uint64_t& s)
{
    const double u1 = 1.0 - (double)(splitmix(s) >> 11) * (1.0 / 9007199254740992.0);
    const double u2 = (double)(splitmix(s) >> 11) * (1.0 / 9007199254740992.0);
    return sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2);
}

}  // namespace sw1dnn

using namespace sw1dnn;

namespace {
thread_local std::string g_nn_err;
int nn_fail(int code, const char* msg, hipError_t e = hipSuccess)
{
    g_nn_err = msg;
    if (e != hipSuccess) g_nn_err += std::string(": ") + hipGetErrorString(e);
    // reported here, so not once more by the next call's launches
    if (code == SW1D_EDEVICE || code == SW1D_ENOMEM) (void)hipGetLastError();
    return code;
}
#define NN_HIP(expr)                                          \
    do {                                                      \
        hipError_t e_ = (expr);                               \
        if (e_ != hipSuccess) return nn_fail(SW1D_EDEVICE, #expr, e_); \
    } while (0)
int g_mfma_ok = 0;
}  // namespace

struct sw1d_nn {
    int X = 1024, Bmax = 0;
    int cus = 256;          // compute units of the device
    int infer_mode = 0;     // 0 auto, 1 per-layer launches, 2 whole-network kernel
    double in_scale = 1.0, out_scale = 1.0;
    hipStream_t stream = nullptr;
    sw1d::HostStage stage;  // host copies of inputs and results
    void* arrays = nullptr;  // the one allocation that the arrays below lie in
    float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;  // NPARAM each
    int64_t adam_t = 0;
    __bf16 *wf[4] = {}, *wb[4] = {};                                // packed mid weights
    float* x = nullptr;     // [B][X] input
    float* du = nullptr;    // [B][X] output
    float* tgt = nullptr;   // [B][X] target
    float* gdu = nullptr;   // [B][X] d loss / d du
    f32x4* Z[4] = {};       // pre-activations of L2..L5, accumulator order
    __bf16* A[2] = {};      // [B][X][C] activations, layers in turn
    __bf16* AT[4] = {};     // [B][C][xt(X)] activations of L1..L4
    __bf16* dZ[2] = {};     // [B][X][C] gradients, layers in turn
    __bf16* dZT[4] = {};    // [B][C][X] gradients of L2..L5
    float* part = nullptr;  // partial gradients of the weight kernel's shares
    float* lossp = nullptr;
    float* taps = nullptr;  // [5][B][X] output-layer tap sums (inference)
    int* keep = nullptr;    // [B] judged-step selection
    double* jacc = nullptr; // [2] judge accumulators over a call: fallbacks, largest error
    // surrogate integration scratch, allocations of its own
    double* usave = nullptr;
    double* unn = nullptr;
    double* l2p = nullptr;
    int64_t int_len = 0;
    // training set (sw1d_nn_dataset)
    float* data_x = nullptr;
    float* data_t = nullptr;
    int64_t data_samples = 0;
};

namespace {

int pack_weights(sw1d_nn* N)
{
    PackOut o;
    for (int l = 0; l < 4; ++l) {
        o.wf[l] = N->wf[l];
        o.wb[l] = N->wb[l];
    }
    hipLaunchKernelGGL(k_pack_w, dim3(nblk(TAPS * C * C), 4), dim3(NT), 0, N->stream, N->p, o);
    NN_HIP(hipGetLastError());
    return SW1D_OK;
}

const float* mid_bias(const sw1d_nn* N, int l) { return N->p + P_MID + l * MID_SZ + TAPS * C * C; }

// Layers 1-5 of B samples from `in` (normalised by inv_scale); the layer-5
// activation ends in N->A[1].  TRAIN keeps what nn_backward needs.
template <int TF, typename TIN, bool TRAIN>
int nn_layers(sw1d_nn* N, int B, const TIN* in, float inv_scale)
{
    const int X = N->X, NTL = Tile<TF>::NT;
    const dim3 grid(X / TF, B);
    hipLaunchKernelGGL((k_l12_fwd<TF, TIN, TRAIN>), grid, dim3(NTL), 0, N->stream, in, inv_scale, N->p + P_W1,
                       N->p + P_B1, N->wf[0], mid_bias(N, 0), N->AT[0], N->Z[0], N->AT[1], N->A[0], X);
    for (int l = 1; l < 4; ++l)
        hipLaunchKernelGGL((k_mid_fwd<TF, TRAIN>), grid, dim3(NTL), 0, N->stream, N->A[(l - 1) & 1], N->wf[l],
                           mid_bias(N, l), N->Z[l], l < 3 ? N->AT[l + 1] : nullptr, N->A[l & 1], X);
    NN_HIP(hipGetLastError());
    return SW1D_OK;
}

// Positions per workgroup of the whole-network kernel: the fewest microseconds
// for B samples of X positions on `cus` compute units.  A launch lasts as long
// as the CU with most workgroups; measured with 1 .. cap of them side by side
// (cap by LDS).
int net_segment(int64_t B, int64_t X, int cus)
{
    struct Split { int seg, cap; float us[6]; };
    static constexpr Split splits[] = {{128, 5, {0, 18.f, 23.f, 30.f, 38.f, 47.f}}, {256, 3, {0, 23.f, 34.f, 50.f}},
                                       {512, 2, {0, 37.f, 57.f}}};
    int best = 0;
    double least = 0;
    for (const Split& c : splits) {
        if (X % c.seg != 0) continue;
        const int64_t m = (B * (X / c.seg) + cus - 1) / cus;
        const double us = (double)(m / c.cap) * c.us[c.cap] + c.us[m % c.cap];
        if (best == 0 || us < least) {
            least = us;
            best = c.seg;
        }
    }
    return best;
}

template <typename TIN, int SEG, int PB>
void launch_net(sw1d_nn* N, int B, const TIN* in, float inv_scale, double* out)
{
    const MidWeights w{{N->wf[0], N->wf[1], N->wf[2], N->wf[3]}};
    hipLaunchKernelGGL((k_net_fwd<TIN, SEG, PB>), dim3((unsigned)((int64_t)B * (N->X / SEG))), dim3(4 * SEG / PB), 0,
                       N->stream, in, inv_scale, N->p, w, N->du, out, N->out_scale, N->X);
}
template <typename TIN>
void net_forward(sw1d_nn* N, int B, const TIN* in, float inv_scale, double* out)
{
    switch (net_segment(B, N->X, N->cus)) {
    case 128: return launch_net<TIN, 128, 2>(N, B, in, inv_scale, out);
    case 256: return launch_net<TIN, 256, 2>(N, B, in, inv_scale, out);
    default: return launch_net<TIN, 512, 4>(N, B, in, inv_scale, out);
    }
}

// Inference of B samples.  u == nullptr: from the FP32 inputs in N->x to du
// in N->du.  Otherwise from the FP64 states u (normalised on the fly by
// 1/in_scale) to out = u + out_scale * du, another array.  One launch of the
// whole-network kernel where nx is a multiple of 256 (2048, 128 samples: 60 us
// against 98; 512, 8 samples: 19 against 33), or five launches (infer_mode = 1), these two with the same bits;
// otherwise 64-position tiles and the training's output layer.
int nn_infer(sw1d_nn* N, int B, const double* u, double* out)
{
    const int X = N->X;
    const int64_t plane = (int64_t)B * X;
    if (X % TILE_F == 0 && N->infer_mode != 1) {
        if (u)
            net_forward<double>(N, B, u, (float)(1.0 / N->in_scale), out);
        else
            net_forward<float>(N, B, N->x, 1.0f, nullptr);
        NN_HIP(hipGetLastError());
        return SW1D_OK;
    }
    if (X % TILE_F != 0) {
        const int rc = u ? nn_layers<TILE, double, false>(N, B, u, (float)(1.0 / N->in_scale))
                         : nn_layers<TILE, float, false>(N, B, N->x, 1.0f);
        if (rc) return rc;
        hipLaunchKernelGGL(k_l6_fwd<false>, dim3(nblk(plane)), dim3(NT), 0, N->stream, N->A[1], N->p + P_W6,
                           N->p + P_B6, N->du, nullptr, nullptr, nullptr, X, plane);
        if (u)
            hipLaunchKernelGGL(k_apply_du, dim3(nblk(plane)), dim3(NT), 0, N->stream, u, N->du, out, plane,
                               N->out_scale);
        NN_HIP(hipGetLastError());
        return SW1D_OK;
    }
    const dim3 grid(X / TILE_F, B);
    const float* P = N->p;
    if (u)
        hipLaunchKernelGGL((k_l12_fwd<TILE_F, double, false>), grid, dim3(NTW), 0, N->stream, u,
                           (float)(1.0 / N->in_scale), P + P_W1, P + P_B1, N->wf[0], mid_bias(N, 0), nullptr, nullptr,
                           nullptr, N->A[0], X);
    else
        hipLaunchKernelGGL((k_l12_fwd<TILE_F, float, false>), grid, dim3(NTW), 0, N->stream, N->x, 1.0f, P + P_W1,
                           P + P_B1, N->wf[0], mid_bias(N, 0), nullptr, nullptr, nullptr, N->A[0], X);
    for (int l = 1; l <= 2; ++l)
        hipLaunchKernelGGL((k_mid_fwd<TILE_F, false>), grid, dim3(NTW), 0, N->stream, N->A[(l - 1) & 1], N->wf[l],
                           mid_bias(N, l), nullptr, nullptr, N->A[l & 1], X);
    hipLaunchKernelGGL(k_l56_fwd, grid, dim3(NTW), 0, N->stream, N->A[0], N->wf[3], mid_bias(N, 3), P + P_W6, N->taps,
                       X, plane);
    if (u)
        hipLaunchKernelGGL(k_l6_out<true>, dim3(nblk(plane)), dim3(NT), 0, N->stream, N->taps, P + P_B6,
                           nullptr, u, out, N->out_scale, X, plane);
    else
        hipLaunchKernelGGL(k_l6_out<false>, dim3(nblk(plane)), dim3(NT), 0, N->stream, N->taps, P + P_B6,
                           N->du, nullptr, nullptr, 0.0, X, plane);
    NN_HIP(hipGetLastError());
    return SW1D_OK;
}

// loss (mean square against N->tgt) of the samples in N->x and the full
// gradient into N->g
template <int TF>
int nn_gradient(sw1d_nn* N, int B)
{
    const int X = N->X, NTL = Tile<TF>::NT;
    const int64_t nout = (int64_t)B * X;
    const dim3 tiles(X / TF, B);
    const int rc = nn_layers<TF, float, true>(N, B, N->x, 1.0f);
    if (rc) return rc;
    hipLaunchKernelGGL(k_l6_fwd<true>, dim3(nblk(nout)), dim3(NT), 0, N->stream, N->A[1], N->p + P_W6, N->p + P_B6,
                       nullptr, N->tgt, N->gdu, N->lossp, X, nout);
    hipLaunchKernelGGL(k_l6_bwd_data<TF>, tiles, dim3(NTL), 0, N->stream, N->gdu, N->p + P_W6, N->Z[3], N->dZT[3],
                       N->dZ[1], X);
    for (int l = 3; l >= 1; --l)
        hipLaunchKernelGGL((k_mid_bwd_data<TF, false>), tiles, dim3(NTL), 0, N->stream, N->dZ[l & 1], N->wb[l],
                           N->Z[l - 1], nullptr, nullptr, nullptr, N->dZT[l - 1], N->dZ[(l - 1) & 1], X);
    hipLaunchKernelGGL((k_mid_bwd_data<TF, true>), tiles, dim3(NTL), 0, N->stream, N->dZ[0], N->wb[0], nullptr, N->x,
                       N->p + P_W1, N->p + P_B1, nullptr, N->dZ[1], X);
    GradIn in;
    for (int l = 0; l < 4; ++l) {
        in.dzt[l] = N->dZT[l];
        in.at[l] = N->AT[l];
    }
    in.g = N->gdu;
    in.a5 = N->A[1];
    in.dz1 = N->dZ[1];
    in.in = N->x;
    const int groups = (int)(nout / 32);
    const int most = groups / 4 > 0 ? groups / 4 : 1;
    const int mids = std::min(MID_SHARES, most), edges = std::min(EDGE_SHARES, most);
    hipLaunchKernelGGL(k_grad_weights, dim3(4 * mids + 2 * edges), dim3(NTG), 0, N->stream, in, N->part, X, groups, mids,
                       edges);
    hipLaunchKernelGGL(k_reduce_grad, dim3(nblk(NPARAM)), dim3(NT), 0, N->stream, N->part, mids, edges, N->g);
    NN_HIP(hipGetLastError());
    return SW1D_OK;
}

// ... and the loss, and the gradient to the host, where asked for
int nn_gradient(sw1d_nn* N, int B, double* loss, float* grad_host = nullptr)
{
    const int rc = N->X % TILE_F == 0 ? nn_gradient<TILE_F>(N, B) : nn_gradient<TILE>(N, B);
    if (rc || (!loss && !grad_host)) return rc;
    const int64_t nout = (int64_t)B * N->X;
    std::vector<float> lp(loss ? nblk(nout) : 0);
    hipError_t e = hipSuccess;
    if (loss) e = N->stage.down(lp.data(), N->lossp, lp.size() * sizeof(float), N->stream);
    if (grad_host && e == hipSuccess) e = N->stage.down(grad_host, N->g, NPARAM * sizeof(float), N->stream);
    const hipError_t done = N->stage.finish(N->stream);  // in any case: lp ends here
    NN_HIP(e);
    NN_HIP(done);
    if (loss) {
        double s = 0;
        for (float f : lp) s += f;
        *loss = s / (double)nout;
    }
    return SW1D_OK;
}

int adam(sw1d_nn* N, float lr, float b1, float b2, float eps)
{
    N->adam_t += 1;
    const float c1 = 1.f - powf(b1, (float)N->adam_t), c2 = 1.f - powf(b2, (float)N->adam_t);
    hipLaunchKernelGGL(k_adam, dim3(nblk(NPARAM)), dim3(NT), 0, N->stream, N->p, N->g, N->m, N->v,
                       NPARAM, lr, b1, b2, eps, c1, c2);
    NN_HIP(hipGetLastError());
    return pack_weights(N);
}

void nn_release(sw1d_nn* N)
{
    if (!N) return;
    if (N->stream) (void)hipStreamSynchronize(N->stream);
    for (void* q : {N->arrays, (void*)N->usave, (void*)N->unn, (void*)N->l2p, (void*)N->data_x, (void*)N->data_t})
        if (q) (void)hipFree(q);
    if (N->stream) (void)hipStreamDestroy(N->stream);
    delete N;
}

template <typename T>
hipError_t dalloc(T** p, size_t count)
{
    return hipMalloc((void**)p, count * sizeof(T));
}

// The network's arrays in one allocation that starts at `base` (null: only its size,
// which is returned), each large one where an allocation of its own would start.
// (64 samples of 1024 positions: created in 1.9 ms and destroyed in 0.5, where 33
// allocations took 2.2 and 3.1.)
size_t lay_out(sw1d_nn* N, char* base)
{
    const size_t nout = (size_t)N->X * N->Bmax, nfeat = nout * C;
    size_t at = 0;
    auto place = [&](auto*& p, size_t count) {
        using T = std::remove_reference_t<decltype(*p)>;
        const size_t bytes = count * sizeof(T), align = bytes >= (1u << 20) ? 1u << 21 : 1u << 12;
        at = (at + align - 1) & ~(align - 1);
        if (base) p = reinterpret_cast<T*>(base + at);
        at += bytes;
    };
    for (int l = 0; l < 4; ++l) {
        place(N->Z[l], nfeat / 4);
        place(N->dZT[l], nfeat);
        place(N->AT[l], (size_t)N->Bmax * C * xt(N->X));
    }
    for (int l = 0; l < 2; ++l) {
        place(N->A[l], nfeat);
        place(N->dZ[l], nfeat);
    }
    place(N->part, WG_SHARES * NPARAM);
    place(N->taps, TAPS * nout);
    for (float** p : {&N->x, &N->du, &N->tgt, &N->gdu}) place(*p, nout);
    for (float** p : {&N->p, &N->g, &N->m, &N->v}) place(*p, NPARAM);
    for (int l = 0; l < 4; ++l) {
        place(N->wf[l], TAPS * C * C);
        place(N->wb[l], TAPS * C * C);
    }
    place(N->lossp, nblk((int64_t)nout));
    place(N->keep, (size_t)N->Bmax);
    place(N->jacc, 2);
    return at;
}

}  // namespace

extern "C" {

const char* sw1d_nn_last_error(void) { return g_nn_err.c_str(); }

int sw1d_nn_param_count(void) { return (int)NPARAM; }

int sw1d_nn_device_check(void)
{
    int* d = nullptr;
    NN_HIP(hipMalloc(&d, sizeof(int)));
    const int one = 1;
    int ok = 0;
    hipError_t e = hipMemcpy(d, &one, sizeof(int), hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_mfma_check, dim3(1), dim3(64), 0, 0, d);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(&ok, d, sizeof(int), hipMemcpyDeviceToHost);
    (void)hipFree(d);
    if (e != hipSuccess) return nn_fail(SW1D_EDEVICE, "MFMA layout check", e);
    g_mfma_ok = ok ? 1 : -1;
    return ok;
}

int sw1d_nn_create(sw1d_nn** out, int32_t nx, int32_t max_batch, uint64_t seed)
{
    if (!out) return nn_fail(SW1D_EINVAL, "null argument");
    *out = nullptr;
    if (nx < TILE || nx % TILE != 0 || nx > (1 << 24) || max_batch < 1 || max_batch > 65535)
        return nn_fail(SW1D_EINVAL, "nx must be a multiple of 64 in [64, 2^24] and 1 <= max_batch <= 65535");
    if (g_mfma_ok == 0 && sw1d_nn_device_check() < 0) return SW1D_EDEVICE;
    if (g_mfma_ok != 1) return nn_fail(SW1D_EDEVICE, "MFMA operand layout check failed on this device");
    sw1d_nn* N = new sw1d_nn();
    N->X = nx;
    N->Bmax = max_batch;
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && cus > 0)
        N->cus = cus;
    const int64_t nout = (int64_t)nx * max_batch;
    // two inputs, the loss parts and the gradient
    N->stage.reserve((size_t)(2 * nout + nblk(nout) + NPARAM) * sizeof(float) + 4 * 4096);
    const size_t bytes = lay_out(N, nullptr);
    const bool ok = hipStreamCreateWithFlags(&N->stream, hipStreamNonBlocking) == hipSuccess &&
                    hipMalloc(&N->arrays, bytes) == hipSuccess;
    if (!ok) {
        nn_release(N);
        return nn_fail(SW1D_ENOMEM, "surrogate device allocation failed");
    }
    lay_out(N, static_cast<char*>(N->arrays));
    // He-style initialisation (std sqrt(2/fan_in)); the output layer starts at
    // zero so the untrained network predicts du = 0.
    std::vector<float> h(NPARAM, 0.f);
    uint64_t s = seed;
    for (int64_t i = 0; i < C * TAPS; ++i) h[P_W1 + i] = (float)(normal(s) * sqrt(2.0 / TAPS));
    for (int l = 0; l < 4; ++l)
        for (int64_t i = 0; i < TAPS * C * C; ++i)
            h[P_MID + l * MID_SZ + i] = (float)(normal(s) * sqrt(2.0 / (TAPS * C)));
    // on the network's stream, which the null stream does not wait for
    hipError_t e = hipMemcpyAsync(N->p, h.data(), NPARAM * sizeof(float), hipMemcpyHostToDevice, N->stream);
    if (e == hipSuccess) e = hipMemsetAsync(N->m, 0, NPARAM * sizeof(float), N->stream);
    if (e == hipSuccess) e = hipMemsetAsync(N->v, 0, NPARAM * sizeof(float), N->stream);
    const hipError_t done = hipStreamSynchronize(N->stream);  // h ends here
    if (e == hipSuccess) e = done;
    if (e != hipSuccess) {
        nn_release(N);
        return nn_fail(SW1D_EDEVICE, "surrogate initialisation", e);
    }
    if (pack_weights(N) != SW1D_OK || hipStreamSynchronize(N->stream) != hipSuccess) {
        nn_release(N);
        return SW1D_EDEVICE;
    }
    *out = N;
    return SW1D_OK;
}

int sw1d_nn_destroy(sw1d_nn* N)
{
    nn_release(N);
    return SW1D_OK;
}

int sw1d_nn_set_scales(sw1d_nn* N, double in_scale, double out_scale)
{
    if (!N || !(in_scale > 0) || !(out_scale > 0)) return nn_fail(SW1D_EINVAL, "scales must be positive");
    N->in_scale = in_scale;
    N->out_scale = out_scale;
    return SW1D_OK;
}

int sw1d_nn_set_inference(sw1d_nn* N, int32_t mode)
{
    if (!N || mode < 0 || mode > 2) return nn_fail(SW1D_EINVAL, "inference mode must be 0, 1 or 2");
    if (mode == 2 && N->X != 1024) return nn_fail(SW1D_EINVAL, "the whole-network kernel needs nx = 1024");
    if (mode == 1 && N->X % TILE_F != 0)
        return nn_fail(SW1D_EINVAL, "the per-layer inference kernels need nx to be a multiple of 256");
    N->infer_mode = mode;
    return SW1D_OK;
}

int sw1d_nn_get_params(sw1d_nn* N, float* host)
{
    if (!N || !host) return nn_fail(SW1D_EINVAL, "null argument");
    NN_HIP(hipMemcpyAsync(host, N->p, NPARAM * sizeof(float), hipMemcpyDeviceToHost, N->stream));
    NN_HIP(hipStreamSynchronize(N->stream));
    return SW1D_OK;
}

int sw1d_nn_set_params(sw1d_nn* N, const float* host)
{
    if (!N || !host) return nn_fail(SW1D_EINVAL, "null argument");
    NN_HIP(hipMemcpyAsync(N->p, host, NPARAM * sizeof(float), hipMemcpyHostToDevice, N->stream));
    int rc = pack_weights(N);
    if (rc) return rc;
    NN_HIP(hipStreamSynchronize(N->stream));
    return SW1D_OK;
}

// y = net(x) for `batch` samples of nx values (normalised units).
int sw1d_nn_forward(sw1d_nn* N, const float* x_host, int32_t batch, float* y_host)
{
    if (!N || !x_host || !y_host) return nn_fail(SW1D_EINVAL, "null argument");
    if (batch < 1 || batch > N->Bmax) return nn_fail(SW1D_EINVAL, "batch out of range");
    const size_t bytes = (size_t)batch * N->X * sizeof(float);
    NN_HIP(N->stage.up(N->x, x_host, bytes, N->stream));
    int rc = nn_infer(N, batch, nullptr, nullptr);
    if (rc) return rc;
    NN_HIP(N->stage.down(y_host, N->du, bytes, N->stream));
    NN_HIP(N->stage.finish(N->stream));
    return SW1D_OK;
}

// Mean-square loss against t and its gradient with respect to every parameter.
int sw1d_nn_gradient(sw1d_nn* N, const float* x_host, const float* t_host, int32_t batch, double* loss,
                     float* grad_host)
{
    if (!N || !x_host || !t_host || !loss) return nn_fail(SW1D_EINVAL, "null argument");
    if (batch < 1 || batch > N->Bmax) return nn_fail(SW1D_EINVAL, "batch out of range");
    const size_t bytes = (size_t)batch * N->X * sizeof(float);
    NN_HIP(N->stage.up(N->x, x_host, bytes, N->stream));
    NN_HIP(N->stage.up(N->tgt, t_host, bytes, N->stream));
    return nn_gradient(N, batch, loss, grad_host);
}

// Adam on device-resident samples: inputs and targets are [nsamples][nx]
// FP32 device arrays (normalised units).  Mini-batches are drawn with a seeded
// generator on the host and gathered on the device.
int sw1d_nn_train(sw1d_nn* N, const float* d_inputs, const float* d_targets, int64_t nsamples,
                  int32_t batch, int64_t iters, float lr, uint64_t seed, double* last_loss)
{
    if (!N || !d_inputs || !d_targets) return nn_fail(SW1D_EINVAL, "null argument");
    if (batch < 1 || batch > N->Bmax || nsamples < 1 || iters < 0)
        return nn_fail(SW1D_EINVAL, "bad batch / sample count");
    if (iters == 0) {
        if (last_loss) *last_loss = 0.0;
        return SW1D_OK;
    }
    // every mini-batch's sample indices, drawn up front and gathered on the device
    std::vector<int64_t> idx((size_t)(iters * batch));
    uint64_t s = seed;
    for (auto& k : idx) k = (int64_t)(splitmix(s) % (uint64_t)nsamples);
    int64_t* didx = nullptr;
    NN_HIP(hipMalloc((void**)&didx, idx.size() * sizeof(int64_t)));
    int rc = hipMemcpyAsync(didx, idx.data(), idx.size() * sizeof(int64_t), hipMemcpyHostToDevice,
                            N->stream) == hipSuccess ? SW1D_OK : nn_fail(SW1D_EDEVICE, "index upload");
    double loss = 0;
    const int64_t n = (int64_t)batch * N->X;
    for (int64_t it = 0; it < iters && !rc; ++it) {
        hipLaunchKernelGGL(k_gather, dim3(nblk(n)), dim3(NT), 0, N->stream, d_inputs, d_targets,
                           didx + it * batch, N->x, N->tgt, N->X, n);
        rc = nn_gradient(N, batch, (it == iters - 1 || it % 50 == 0) ? &loss : nullptr);
        if (!rc) rc = adam(N, lr, 0.9f, 0.999f, 1e-8f);
    }
    if (hipStreamSynchronize(N->stream) != hipSuccess && !rc) rc = nn_fail(SW1D_EDEVICE, "training");
    (void)hipFree(didx);
    if (rc) return rc;
    if (last_loss) *last_loss = loss;
    return SW1D_OK;
}

}  // extern "C"

// ===================================================== surrogate integrator ===
#include "sw1d_internal.hpp"

extern "C" int sw1d_surrogate_advance(sw1d_nn* N, sw1d_batch* batch, int64_t surrogate_steps,
                                      int32_t k_steps, int32_t judge_every, double tol, double* stats)
{
    sw1d::BatchView bv;
    if (!N || !sw1d::batch_view(batch, bv)) return nn_fail(SW1D_EINVAL, "null argument");
    if (!bv.f64 || !bv.all_ks || bv.n != N->X)
        return nn_fail(SW1D_EINVAL, "surrogate batches hold FP64 KS problems of the network's nx");
    if (bv.count > N->Bmax) return nn_fail(SW1D_EINVAL, "batch larger than the network's max_batch");
    if (k_steps < 1 || surrogate_steps < 0) return nn_fail(SW1D_EINVAL, "bad step counts");
    const int64_t B = bv.count, X = N->X, len = B * X;
    const unsigned blocks = nblk(len);
    const int64_t per = (X + NT - 1) / NT;  // l2 blocks per problem
    if (N->int_len < len) {
        if (N->usave) (void)hipFree(N->usave);
        if (N->unn) (void)hipFree(N->unn);
        if (N->l2p) (void)hipFree(N->l2p);
        N->usave = N->unn = N->l2p = nullptr;
        N->int_len = 0;  // also where an allocation fails
        if (dalloc(&N->usave, len) != hipSuccess || dalloc(&N->unn, len) != hipSuccess ||
            dalloc(&N->l2p, 2 * per * B) != hipSuccess)
            return nn_fail(SW1D_ENOMEM, "integrator scratch");
        N->int_len = len;
    }
    // The states alternate between the batch's array u and the scratch array; a
    // judged step finds its input in u, where the plain solver starts from it.
    double* u = static_cast<double*>(bv.state);
    double *cur = u, *other = N->usave;
    const size_t bytes = (size_t)len * sizeof(double);
    int64_t judged = 0;
    // The judge runs in stream order: the plain solver on the batch's stream
    // waits for the network step (event a), the decision on the network's
    // stream waits for the plain solver (event b); N->jacc accumulates the
    // fallback count and the largest judged error over the call.
    struct Events {
        hipEvent_t a = nullptr, b = nullptr;
        ~Events()
        {
            if (a) (void)hipEventDestroy(a);
            if (b) (void)hipEventDestroy(b);
        }
    } ev;
    NN_HIP(hipEventCreateWithFlags(&ev.a, hipEventDisableTiming));
    NN_HIP(hipEventCreateWithFlags(&ev.b, hipEventDisableTiming));
    NN_HIP(hipStreamSynchronize(bv.stream));
    hipLaunchKernelGGL(k_zero_f64, dim3(1), dim3(NT), 0, N->stream, N->jacc, (int64_t)2);
    auto step = [&](int64_t i) -> int {
        const bool judge = judge_every > 0 && i % judge_every == 0;
        int rc = nn_infer(N, (int)B, cur, judge ? N->unn : other);
        if (rc) return rc;
        if (!judge) {
            std::swap(cur, other);
            return SW1D_OK;
        }
        // plain solver from the same states: u <- solver^K(u)
        if (cur != u) {
            NN_HIP(hipMemcpyAsync(u, cur, bytes, hipMemcpyDeviceToDevice, N->stream));
            std::swap(cur, other);
        }
        NN_HIP(hipEventRecord(ev.a, N->stream));
        NN_HIP(hipStreamWaitEvent(bv.stream, ev.a, 0));
        ++judged;
        rc = sw1d_batch_advance(batch, k_steps);
        if (rc) return nn_fail(rc, "plain solver step of the judge");
        NN_HIP(hipEventRecord(ev.b, bv.stream));
        NN_HIP(hipStreamWaitEvent(N->stream, ev.b, 0));
        hipLaunchKernelGGL(k_l2_parts, dim3((unsigned)per, (unsigned)B), dim3(NT), 0, N->stream, N->unn, u, (int)X,
                           N->l2p);
        hipLaunchKernelGGL(k_judge, dim3(1), dim3(NT), 0, N->stream, N->l2p, B, per, tol, N->keep, N->jacc);
        hipLaunchKernelGGL(k_keep_rows, dim3(blocks), dim3(NT), 0, N->stream, u, N->unn, N->keep, (int)X, len);
        NN_HIP(hipGetLastError());
        return SW1D_OK;
    };
    int rc = SW1D_OK;
    for (int64_t i = 1; i <= surrogate_steps && !rc; ++i) rc = step(i);
    // the batch holds the last step that was taken, also where the next one failed
    if (cur != u) {
        const hipError_t e = hipMemcpyAsync(u, cur, bytes, hipMemcpyDeviceToDevice, N->stream);
        if (e != hipSuccess && !rc) rc = nn_fail(SW1D_EDEVICE, "states into the batch", e);
    }
    if (rc) {
        (void)hipStreamSynchronize(N->stream);
        return rc;
    }
    double acc[2] = {0.0, 0.0};
    NN_HIP(hipMemcpyAsync(acc, N->jacc, sizeof(acc), hipMemcpyDeviceToHost, N->stream));
    NN_HIP(hipStreamSynchronize(N->stream));
    const int64_t fallbacks = (int64_t)acc[0];
    const double max_err = acc[1];
    if (stats) {
        stats[0] = (double)surrogate_steps;
        stats[1] = (double)judged;
        stats[2] = (double)fallbacks;
        stats[3] = max_err;
    }
    return SW1D_OK;
}

// ============================================================ training data ===
namespace sw1dnn {
// x = u_s / in_scale, t = (u_{s+1} - u_s) / out_scale for one snapshot pair
__global__ __launch_bounds__(NT) void k_make_pairs(const double* __restrict__ u0, const double* __restrict__ u1,
                                                   float* __restrict__ x, float* __restrict__ t, int64_t n,
                                                   double inv_in, double inv_out)
{
    const int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x;
    if (i >= n) return;
    x[i] = (float)(u0[i] * inv_in);
    t[i] = (float)((u1[i] - u0[i]) * inv_out);
}
// partial sums of a^2 and (b-a)^2
__global__ __launch_bounds__(NT) void k_sq_parts(const double* __restrict__ a, const double* __restrict__ b,
                                                 int64_t n, double* __restrict__ part)
{
    __shared__ double r0[NT], r1[NT];
    const int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x;
    double s0 = 0, s1 = 0;
    if (i < n) {
        s0 = a[i] * a[i];
        s1 = (b[i] - a[i]) * (b[i] - a[i]);
    }
    r0[threadIdx.x] = s0;
    r1[threadIdx.x] = s1;
    __syncthreads();
    for (int k = NT / 2; k > 0; k >>= 1) {
        if (threadIdx.x < k) {
            r0[threadIdx.x] += r0[threadIdx.x + k];
            r1[threadIdx.x] += r1[threadIdx.x + k];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = r0[0];
        part[2 * blockIdx.x + 1] = r1[0];
    }
}
}  // namespace sw1dnn

extern "C" {

void sw1d_nn_release_dataset(sw1d_nn* N)
{
    if (!N) return;
    if (N->data_x) (void)hipFree(N->data_x);
    if (N->data_t) (void)hipFree(N->data_t);
    N->data_x = N->data_t = nullptr;
    N->data_samples = 0;
}

// Build the training set from an FP64 KS batch: advance it nsnap times by
// k_steps, keep every snapshot, and store the normalised pairs in the network
// (in_scale = RMS of u, out_scale = RMS of the K-step change).
int sw1d_nn_dataset(sw1d_nn* N, sw1d_batch* batch, int32_t nsnap, int32_t k_steps, int64_t* nsamples,
                    double* scales)
{
    sw1d::BatchView bv;
    if (!N || !sw1d::batch_view(batch, bv) || nsnap < 1 || k_steps < 1)
        return nn_fail(SW1D_EINVAL, "bad dataset arguments");
    if (!bv.f64 || !bv.all_ks || bv.n != N->X)
        return nn_fail(SW1D_EINVAL, "datasets come from FP64 KS batches of the network's nx");
    const int64_t len = bv.count * bv.n;
    const size_t bytes = (size_t)len * sizeof(double);
    double* raw = nullptr;
    if (hipMalloc((void**)&raw, bytes * (size_t)(nsnap + 1)) != hipSuccess)
        return nn_fail(SW1D_ENOMEM, "snapshot storage");
    int rc = SW1D_OK;
    // Snapshots in the order of the batch's own stream: a plain copy between device
    // memories returns before it is done, and the null stream that it runs on waits
    // for no stream of the library's.
    for (int s = 0; s <= nsnap && rc == SW1D_OK; ++s) {
        if (s > 0) rc = sw1d_batch_advance(batch, k_steps);
        if (rc == SW1D_OK && hipMemcpyAsync(raw + (size_t)s * len, bv.state, bytes, hipMemcpyDeviceToDevice,
                                            bv.stream) != hipSuccess)
            rc = SW1D_EDEVICE;
    }
    if (hipStreamSynchronize(bv.stream) != hipSuccess && rc == SW1D_OK) rc = SW1D_EDEVICE;
    const unsigned blocks = nblk(len);
    std::vector<double> parts(2 * (size_t)blocks);
    double* dparts = nullptr;
    double su = 0, sd = 0;
    if (rc == SW1D_OK && hipMalloc((void**)&dparts, parts.size() * sizeof(double)) != hipSuccess) rc = SW1D_ENOMEM;
    for (int s = 0; s < nsnap && rc == SW1D_OK; ++s) {
        hipLaunchKernelGGL(k_sq_parts, dim3(blocks), dim3(NT), 0, N->stream, raw + (size_t)s * len,
                           raw + (size_t)(s + 1) * len, len, dparts);
        if (hipMemcpyAsync(parts.data(), dparts, parts.size() * sizeof(double), hipMemcpyDeviceToHost,
                           N->stream) != hipSuccess || hipStreamSynchronize(N->stream) != hipSuccess)
            rc = SW1D_EDEVICE;
        for (size_t k = 0; k < blocks; ++k) { su += parts[2 * k]; sd += parts[2 * k + 1]; }
    }
    const double cnt = (double)len * nsnap, in_scale = sqrt(su / cnt), out_scale = sqrt(sd / cnt);
    const bool replaced = rc == SW1D_OK;
    if (replaced) {
        sw1d_nn_release_dataset(N);
        N->data_samples = (int64_t)nsnap * bv.count;
        if (dalloc(&N->data_x, (size_t)len * nsnap) != hipSuccess ||
            dalloc(&N->data_t, (size_t)len * nsnap) != hipSuccess)
            rc = SW1D_ENOMEM;
    }
    for (int s = 0; s < nsnap && rc == SW1D_OK; ++s)
        hipLaunchKernelGGL(k_make_pairs, dim3(blocks), dim3(NT), 0, N->stream, raw + (size_t)s * len,
                           raw + (size_t)(s + 1) * len, N->data_x + (size_t)s * len, N->data_t + (size_t)s * len, len,
                           1.0 / in_scale, 1.0 / out_scale);
    if (rc == SW1D_OK && (hipGetLastError() != hipSuccess || hipStreamSynchronize(N->stream) != hipSuccess))
        rc = SW1D_EDEVICE;
    if (dparts) (void)hipFree(dparts);
    (void)hipFree(raw);
    if (rc != SW1D_OK) {
        if (replaced) sw1d_nn_release_dataset(N);  // rather than a part of one
        return nn_fail(rc, "dataset generation failed");
    }
    N->in_scale = in_scale;
    N->out_scale = out_scale;
    if (nsamples) *nsamples = N->data_samples;
    if (scales) { scales[0] = in_scale; scales[1] = out_scale; }
    return SW1D_OK;
}

// Adam on samples [0, nfit) of the stored dataset.
int sw1d_nn_fit(sw1d_nn* N, int64_t nfit, int32_t batch, int64_t iters, float lr, uint64_t seed,
                double* last_loss)
{
    if (!N || !N->data_x) return nn_fail(SW1D_EINVAL, "no dataset (call sw1d_nn_dataset first)");
    if (nfit <= 0 || nfit > N->data_samples) nfit = N->data_samples;
    return sw1d_nn_train(N, N->data_x, N->data_t, nfit, batch, iters, lr, seed, last_loss);
}

// Relative L2 error of the predicted K-step change over samples [first, first+count).
int sw1d_nn_eval(sw1d_nn* N, int64_t first, int64_t count, double* rel_err)
{
    if (!N || !N->data_x || !rel_err) return nn_fail(SW1D_EINVAL, "no dataset or null argument");
    if (first < 0 || count < 1 || first + count > N->data_samples) return nn_fail(SW1D_EINVAL, "range");
    const size_t row = (size_t)N->X;
    double se = 0, st = 0;
    std::vector<float> y, t;
    for (int64_t s = first; s < first + count; s += N->Bmax) {
        const int b = (int)std::min<int64_t>(N->Bmax, first + count - s);
        NN_HIP(hipMemcpyAsync(N->x, N->data_x + s * row, b * row * sizeof(float), hipMemcpyDeviceToDevice, N->stream));
        int rc = nn_infer(N, b, nullptr, nullptr);
        if (rc) return rc;
        y.resize(b * row);
        t.resize(b * row);
        NN_HIP(hipMemcpyAsync(y.data(), N->du, b * row * sizeof(float), hipMemcpyDeviceToHost, N->stream));
        NN_HIP(hipMemcpyAsync(t.data(), N->data_t + s * row, b * row * sizeof(float), hipMemcpyDeviceToHost, N->stream));
        NN_HIP(hipStreamSynchronize(N->stream));
        for (size_t k = 0; k < y.size(); ++k) {
            se += (double)(y[k] - t[k]) * (y[k] - t[k]);
            st += (double)t[k] * t[k];
        }
    }
    *rel_err = sqrt(se / st);
    return SW1D_OK;
}

// Copy stored pairs [first, first+count) to the host (sample s*B + b is
// snapshot s of problem b).  x_host / t_host may be NULL.
int sw1d_nn_dataset_samples(sw1d_nn* N, int64_t first, int64_t count, float* x_host, float* t_host)
{
    if (!N || !N->data_x) return nn_fail(SW1D_EINVAL, "no dataset (call sw1d_nn_dataset first)");
    if (first < 0 || count < 1 || first + count > N->data_samples) return nn_fail(SW1D_EINVAL, "range");
    const size_t row = (size_t)N->X, bytes = (size_t)count * row * sizeof(float);
    if (x_host)
        NN_HIP(hipMemcpyAsync(x_host, N->data_x + first * row, bytes, hipMemcpyDeviceToHost, N->stream));
    if (t_host)
        NN_HIP(hipMemcpyAsync(t_host, N->data_t + first * row, bytes, hipMemcpyDeviceToHost, N->stream));
    NN_HIP(hipStreamSynchronize(N->stream));
    return SW1D_OK;
}

}  // extern "C"
