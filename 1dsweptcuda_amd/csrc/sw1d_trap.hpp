// Device code of Euler's overlapped trapezoid tile (one wave64 per tile,
// sw1d_trapezoid.hip).
//
// A tile's window is 64*PI consecutive points (mod n) starting at `win`;
// lane l holds points l*PI .. l*PI+PI-1 in VGPRs.  After S stages the window
// positions RS .. RS+count-1 (RS = R*S) hold the classic scheme's values and
// are stored to out0 .. out0+count-1 (mod n).
#pragma once

#include "sw1d_euler.hpp"
#include "sw1d_internal.hpp"
#include "sw1d_lanes.hpp"

namespace sw1d {

// i mod n in [0, n).  The tiles' indices lie within one period of the
// domain (window starts in [0, n), windows and output ranges no longer than
// n), so one add or subtract wraps them; the 64-bit remainder, a long
// software sequence on the GPU, is there for any other index and runs only
// in a wave that has one.
__device__ __forceinline__ int64_t wrapn(int64_t i, int64_t n)
{
    if (i >= -n && i < 2 * n) return i < 0 ? i + n : (i >= n ? i - n : i);
    i %= n;
    return i < 0 ? i + n : i;
}

// Lane l's PI window points win + l*PI + p (mod n).  Windows that do not wrap
// (all but the tiles next to the domain ends) index directly.
template <typename T, int PI>
__device__ __forceinline__ void load_window(const T* __restrict__ a, int64_t n, int64_t win,
                                            int lane, T (&v)[PI])
{
    const int64_t i0 = win + (int64_t)lane * PI;
    if (win + (int64_t)kWave * PI <= n) {
#pragma unroll
        for (int p = 0; p < PI; ++p) v[p] = a[i0 + p];
    } else {
#pragma unroll
        for (int p = 0; p < PI; ++p) v[p] = a[wrapn(i0 + p, n)];
    }
}

// Store the points at window positions RS .. RS+count-1 to out0 + (pos - RS).
template <typename T, int PI>
__device__ __forceinline__ void store_window(T* __restrict__ a, int64_t n, int64_t out0, int count,
                                             int lane, int RS, const T (&v)[PI])
{
    const bool direct = out0 + count <= n;
#pragma unroll
    for (int p = 0; p < PI; ++p) {
        const int pos = lane * PI + p - RS;
        if (pos >= 0 && pos < count) a[direct ? out0 + pos : wrapn(out0 + pos, n)] = v[p];
    }
}

// ----------------------------------------------------------------- Euler ---
// One stage (eu_lane_stage): dst = base + c flux(src).  The window's outermost
// cells are discarded, so every stage leaves out their outer interfaces.
template <typename T, int PI, bool BND>
__device__ __forceinline__ void eu_trap_stage(const T (&src)[3][PI], T (&dst)[3][PI],
                                              const T (&base)[3][PI], T (&hl)[3][2], T (&hr)[3][2],
                                              int64_t g0, int64_t n, T c, const EulerCoef<T>& k)
{
    // global index of the lane's cell p, p = -1 .. PI
    auto gidx = [&](int p) {
        const int64_t g = g0 + p;
        return g < 0 ? g + n : (g >= n ? g - n : g);
    };
    // the interface right of cell 0 drops pdiff(-1,0), the one right of cell
    // n-2 drops pdiff(n-1,n) (the flags of Euler:405, :424)
    auto drop0 = [&](int j) { return BND && gidx(j - 1) == 0; };
    auto drop2 = [&](int j) { return BND && gidx(j - 1) == n - 2; };
    eu_lane_stage<false, T, PI>(src, hl, hr, k, drop0, drop2, [&](int p, const Q3<T>& f) {
        Q3<T> nv = eu_apply(Q3<T>{base[0][p], base[1][p], base[2][p]}, f, c);
        if (BND) {  // ghost cells hold the Dirichlet states (Euler:407-416)
            const int64_t g = gidx(p);
            nv = g == 0 ? k.bl : nv;
            nv = g == n - 1 ? k.br : nv;
        }
        dst[0][p] = nv.x;
        dst[1][p] = nv.y;
        dst[2][p] = nv.z;
    });
}

template <typename T, int PI, int S, bool BND>
__device__ __forceinline__ void trap_euler(const T* __restrict__ in, T* __restrict__ out, int64_t n,
                                           int64_t win, int64_t out0, int count, int lane,
                                           const EulerCoef<T>& k)
{
    constexpr int RS = 2 * S;
    T q[3][PI], qh[3][PI];
    const int64_t g0 = wrapn(win + (int64_t)lane * PI, n);
#pragma unroll
    for (int c = 0; c < 3; ++c) load_window<T, PI>(in + c * n, n, win, lane, q[c]);
    const T ca = T(0.25) * k.dtdx, cb = T(0.5) * k.dtdx;
    // beyond the window (discarded cells): the carried registers' values,
    // a physical state so that the discarded cells stay finite
    T hl[3][2], hr[3][2], hlh[3][2], hrh[3][2];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int i = 0; i < 2; ++i) hl[c][i] = hr[c][i] = hlh[c][i] = hrh[c][i] = q[c][0];
    for (int s = 0; s < S; s += 2) {
        eu_trap_stage<T, PI, BND>(q, qh, q, hl, hr, g0, n, ca, k);     // predictor (Euler:307-350)
        eu_trap_stage<T, PI, BND>(qh, q, q, hlh, hrh, g0, n, cb, k);   // corrector (Euler:353-389)
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) store_window<T, PI>(out + c * n, n, out0, count, lane, RS, q[c]);
}


}  // namespace sw1d
