// Overlapped trapezoid tiles of Euler (heat and KS plans run the workgroup-wide
// tiles of sw1d_wide.hip) — the up-triangle of the swept rule with its base
// widened by R*S cells on each side so that after S stages its top is a full
// output tile of W_out = 64*PO cells.
//
// One wave64 per tile.  Lane l holds PI = PO + 1 consecutive cells of the
// W_in = 64*PI cell window in VGPRs; every stage updates every cell of the
// window, neighbours crossing lanes through DPP wave shifts.  A cell's value
// after stage s is exact when its stage-s dependency cone lies inside the
// window, which holds for the W_in - 4*s central cells, so after S = 16 stages
// the W_out central cells are the classic scheme's values, bitwise (same
// formulas, same operands).  The cells nearer the window edges are recomputed
// by the neighbouring tile.
//
// Any nX works: tiles start at multiples of W_out, the last one stores only
// the cells that exist, addresses wrap modulo nX.  The state crossing launches
// is the plain field (rho, m, E) at a full time step.
//
// Tiles whose window touches cell 0 or nX-1 run a variant that carries the
// per-cell checks of the Dirichlet ends; all other tiles run without them.

#include "sw1d_trap.hpp"

namespace sw1d {
namespace {

constexpr int kWavesPerBlock = 4;
constexpr int kBlock = kWave * kWavesPerBlock;

// ---------------------------------------------------------------- kernel ---
template <typename T, int PO>
__global__ __launch_bounds__(kBlock) void k_trapezoid(const T* __restrict__ in, T* __restrict__ out,
                                                      int64_t n, int64_t ntiles, int64_t tile_first,
                                                      EulerCoef<T> eu)
{
    constexpr int PI = PO + 1, WIN = kWave * PI, WOUT = kWave * PO, RS = 32, S = 16;
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t tile = tile_first + (int64_t)blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
    if (tile >= ntiles) return;
    const int64_t out0 = tile * WOUT;
    const int count = (int)(n - out0 < WOUT ? n - out0 : WOUT);
    const int64_t win = wrapn(out0 - RS, n);
    // does the window reach cell 0 or cell n-1?
    const bool bnd = out0 < RS + 1 || out0 - RS + WIN > n - 1 || WIN >= n;
    if (bnd)
        trap_euler<T, PI, S, true>(in, out, n, win, out0, count, lane, eu);
    else
        trap_euler<T, PI, S, false>(in, out, n, win, out0, count, lane, eu);
}

template <typename T, int PO>
hipError_t trap_tile(const TrapLaunch& L, const EulerCoef<T>& eu, hipStream_t s)
{
    const int64_t count = L.ntiles - L.tile_first;
    if (count <= 0) return hipSuccess;
    const dim3 grid((unsigned)((count + kWavesPerBlock - 1) / kWavesPerBlock));
    hipLaunchKernelGGL((k_trapezoid<T, PO>), grid, dim3(kBlock), 0, s, static_cast<const T*>(L.in),
                       static_cast<T*>(L.out), L.n, L.ntiles, L.tile_first, eu);
    return hipGetLastError();
}

template <typename T>
hipError_t trap_prec(const TrapLaunch& L, const EulerCoef<T>& eu, hipStream_t s)
{
    if (L.eq != EQ_EULER || L.SB != 1) return hipErrorInvalidValue;
    if (L.PO == 2) return trap_tile<T, 2>(L, eu, s);
    if (L.PO == 4) return trap_tile<T, 4>(L, eu, s);
    return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_trapezoid(const TrapLaunch& L, bool f64, const Coefs& c, hipStream_t s)
{
    return f64 ? trap_prec<double>(L, c.eu_d, s) : trap_prec<float>(L, c.eu_f, s);
}

bool trapezoid_supported(int eq, int PO, int SB)
{
    if (eq == EQ_EULER) return SB == 1 && (PO == 2 || PO == 4);
    return (SB == 1 && (PO == 2 || PO == 4 || PO == 8 || PO == 16)) ||
           (SB == 2 && (PO == 8 || PO == 16));
}

}  // namespace sw1d
