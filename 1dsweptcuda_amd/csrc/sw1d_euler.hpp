// One Euler stage over a wave whose lane l holds P consecutive cells, shared by
// the swept, trapezoid and wide tiles.
//
// A cell's update needs the fluxes at both its interfaces, an interface is
// some 300 instructions (seven divisions, three square roots), and two cells
// share it.  A lane evaluates the interfaces left of its own cells; the one
// right of its last cell is the next lane's first, which a lane shift brings
// (six values): P interfaces for P cells instead of P + 1, the values of the
// per-cell form, so the same bits.  Pressure differences are shared the same
// way.  At 4 cells per lane and the regions below it that is 29% fewer
// interfaces (Euler diamond at 2^18 cells, W = 256: see k_euler_swept).
#pragma once

#include "sw1d_internal.hpp"
#include "sw1d_lanes.hpp"

namespace sw1d {

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
    auto iface = [&](int j, Q3<T>& F, Q3<T>& D) {
        const T q0 = drop0(j) ? T(0) : pd[j];
        const T q2 = drop2(j) ? T(0) : pd[j + 2];
        const Q3<T> A{e[0][j], T(0), T(0)}, B{e[0][j + 3], T(0), T(0)};  // their densities only
        eu_iface(A, cell(j + 1), cell(j + 2), B, q0, pd[j + 1], q2, k, F, D);
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
}

}  // namespace sw1d
