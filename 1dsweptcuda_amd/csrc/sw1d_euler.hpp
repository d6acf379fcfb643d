// One Euler stage over a wave whose lane l holds P consecutive cells, shared by
// the swept rows, the wide tiles and the classic step.
//
// A cell's update needs the fluxes at both its interfaces, an interface is
// some 300 instructions (seven divisions, three square roots), and two cells
// share it.  A lane evaluates the interfaces left of its own cells; the one
// right of its last cell is the next lane's first, which a lane shift brings
// (six values): P interfaces for P cells instead of P + 1, the values of the
// per-cell form, so the same bits.  Pressure differences are shared the same
// way.  At 4 cells per lane and the regions below it that is 29% fewer
// interfaces (swept tiles of 2^18 cells, W = 256, FP64: 2.95e10 -> 3.84e10
// point-updates/s).
#pragma once

#include "sw1d_internal.hpp"
#include "sw1d_lanes.hpp"

namespace sw1d {

// Quotients and roots of regular operands (eu_regular below) with the bits of
// the operators: Newton-Raphson reciprocals, Goldschmidt's square root and
// Markstein's residual correction, which rounds correctly, without the
// operators' scaling for operands whose intermediates leave the number range.
// A density's reciprocal serves both of its quotients.  An FP64 interface takes
// 240 instructions instead of 281 (the same tiles: 3.84e10 -> 4.26e10
// point-updates/s; 2^20, W = 512: 5.10e10 -> 5.53e10).
template <typename T> struct Quick;
template <> struct Quick<double> {
    struct Den { double b, y; };
    static __device__ __forceinline__ Den over(double b)
    {
        double y = __builtin_amdgcn_rcp(b);
        y = fma(fma(-b, y, 1.0), y, y);
        return Den{b, fma(fma(-b, y, 1.0), y, y)};
    }
    static __device__ __forceinline__ double quot(double a, const Den& d)
    {
        const double q = a * d.y;
        return fma(fma(-d.b, q, a), d.y, q);
    }
    // a may be a zero of either sign
    static __device__ __forceinline__ double div(double a, const Den& d)
    {
        return __builtin_amdgcn_div_fixup(quot(a, d), d.b, a);
    }
    static __device__ __forceinline__ double root(double x)
    {
        const double y = __builtin_amdgcn_rsq(x);
        double g = x * y, h = 0.5 * y;
        const double r = fma(-h, g, 0.5);
        g = fma(g, r, g);
        h = fma(h, r, h);
        g = fma(fma(-g, g, x), h, g);
        return fma(fma(-g, g, x), h, g);
    }
};
template <> struct Quick<float> {
    struct Den { float b, y; };
    static __device__ __forceinline__ Den over(float b)
    {
        const float y = __builtin_amdgcn_rcpf(b);
        return Den{b, fmaf(fmaf(-b, y, 1.0f), y, y)};
    }
    static __device__ __forceinline__ float quot(float a, const Den& d)
    {
        float q = a * d.y;
        q = fmaf(fmaf(-d.b, q, a), d.y, q);
        return fmaf(fmaf(-d.b, q, a), d.y, q);
    }
    static __device__ __forceinline__ float div(float a, const Den& d)
    {
        return __builtin_amdgcn_div_fixupf(quot(a, d), d.b, a);
    }
    static __device__ __forceinline__ float root(float x)
    {
        const float y = __builtin_amdgcn_rsqf(x);
        float g = x * y, h = 0.5f * y;
        const float r = fmaf(-h, g, 0.5f);
        g = fmaf(g, r, g);
        h = fmaf(h, r, h);
        return fmaf(fmaf(-g, g, x), h, g);
    }
};

// Whether a wave's stage may use Quick: every density and energy in [2^-X,
// 2^X), every momentum below 2^X; X = 64 in FP64, 8 in FP32.  The limited
// states lie between their cells, so the densities that are divided by and
// rooted are in that range and a divisor made of them within [2^-2X, 2^2X+2].
// A momentum, and so a velocity, may be any tiny number or zero: below 2^-968
// (FP32 2^-100) the residual of its quotient is not exact, but such a velocity
// times a momentum is zero, and otherwise it is added, as energy flux, to an
// energy of at least 2^-X, which no number so small changes.  A NaN, an
// infinity, a negative density or energy fails the test.  The limiter's
// ratios keep the operator: their operands, pressure differences, fall
// through the whole range of numbers at the foot of every front.
template <typename T> struct Regular;
template <> struct Regular<double> {
    static constexpr uint32_t lo = (1023u - 64) << 20, hi = (1023u + 64) << 20;
    static __device__ __forceinline__ uint32_t bits(double v) { return (uint32_t)__double2hiint(v); }
};
template <> struct Regular<float> {
    static constexpr uint32_t lo = (127u - 8) << 23, hi = (127u + 8) << 23;
    static __device__ __forceinline__ uint32_t bits(float v) { return __float_as_uint(v); }
};
// e: ext cells j0 .. j1 - 1 of a lane
template <typename T, int NE>
__device__ __forceinline__ bool eu_regular(const T (&e)[3][NE], int j0, int j1)
{
    using G = Regular<T>;
    uint32_t most = 0, least = ~0u;
#pragma unroll
    for (int j = j0; j < j1; ++j) {
        const uint32_t a = G::bits(e[0][j]), b = G::bits(e[1][j]) & 0x7fffffffu, c = G::bits(e[2][j]);
        most = max(max(most, a), max(b, c));
        least = min(min(least, a), c);
    }
    return __builtin_amdgcn_ballot_w64(most >= G::hi || least < G::lo) == 0;
}

// v: the lane's cells, component c at v[c][p]; hl / hr: its outer neighbours,
// carried from call to call (gather_carry), nearest first.  The first cell of
// lane 0 and the last of lane 63 have no lane beyond them: with FULL their
// outer interfaces are evaluated too (P + 1 per lane), else the two cells (and
// the neighbour of the last) receive values that the caller does not use.
// drop0(j) / drop2(j): interface j, left of the lane's cell j, has the left
// ghost cell on its left / the right ghost cell on its right and drops the
// pressure difference beyond it.  out(p, f): cell p's net flux.
template <bool FULL, typename T, int P, typename D0, typename D2, typename OUT>
__device__ __forceinline__ void eu_lane_stage(const T (*v)[P], T (*hl)[2], T (*hr)[2], const EulerCoef<T>& k, D0&& drop0,
                                              D2&& drop2, OUT&& out)
{
    T e[3][P + 4];  // ext cell j is the lane's cell j - 2
#pragma unroll
    for (int c = 0; c < 3; ++c) {
#pragma unroll
        for (int p = 0; p < P; ++p) e[c][p + 2] = v[c][p];
        hl[c][0] = from_left(e[c][P + 1], hl[c][0]);
        hr[c][0] = from_right(e[c][2], hr[c][0]);
        e[c][1] = hl[c][0];
        e[c][P + 2] = hr[c][0];
        // the second neighbours: for the limiter of interface 0 the density
        // only
        if (FULL || c == 0) {
            hl[c][1] = from_left(e[c][P], hl[c][1]);
            e[c][0] = hl[c][1];
        }
        if (FULL) {
            hr[c][1] = from_right(e[c][3], hr[c][1]);
            e[c][P + 3] = hr[c][1];
        }
    }
    auto cell = [&](int j) { return Q3<T>{e[0][j], e[1][j], e[2][j]}; };
    T pd[P + 3];  // pressure differences between ext cells j and j + 1
#pragma unroll
    for (int j = 1; j <= P; ++j) pd[j] = eu_pdiff(cell(j), cell(j + 1));
    if (FULL) {
        pd[0] = eu_pdiff(cell(0), cell(1));
        pd[P + 1] = eu_pdiff(cell(P + 1), cell(P + 2));
        pd[P + 2] = eu_pdiff(cell(P + 2), cell(P + 3));
    } else {
        pd[0] = from_left0(pd[P]);
        pd[P + 1] = from_right0(pd[1]);
    }
    auto stage = [&](auto math) {
        using M = decltype(math);
        auto iface = [&](int j, Q3<T>& F, Q3<T>& D) {
            const T q0 = drop0(j) ? T(0) : pd[j];
            const T q2 = drop2(j) ? T(0) : pd[j + 2];
            const Q3<T> A{e[0][j], T(0), T(0)}, B{e[0][j + 3], T(0), T(0)};  // their densities only
            eu_iface<M>(A, cell(j + 1), cell(j + 2), B, q0, pd[j + 1], q2, k, F, D);
        };
        Q3<T> FL, DL, FE, DE;
        iface(0, FL, DL);
        if (FULL) {
            iface(P, FE, DE);
        } else {
            FE = Q3<T>{from_right0(FL.x), from_right0(FL.y), from_right0(FL.z)};
            DE = Q3<T>{from_right0(DL.x), from_right0(DL.y), from_right0(DL.z)};
        }
#pragma unroll
        for (int p = 0; p < P; ++p) {
            Q3<T> FR, DR;
            if (p + 1 < P) {
                iface(p + 1, FR, DR);
            } else {
                FR = FE;
                DR = DE;
            }
            out(p, eu_balance(FL, DL, FR, DR));
            FL = FR;
            DL = DR;
        }
    };
    // the lanes beyond test the neighbours' cells, except those beyond the wave
    const bool regular = FULL ? eu_regular(e, 0, P + 4) : eu_regular(e, 2, P + 2);
    if (regular)
        stage(Quick<T>{});
    else
        stage(Ieee<T>{});
}

}  // namespace sw1d
