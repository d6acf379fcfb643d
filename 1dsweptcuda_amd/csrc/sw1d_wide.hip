// Workgroup-wide overlapped tiles (sw1d_wide.hpp) for single plans: the kernels, and
// the choice of a tile shape and of the steps per launch.
//
// An advance of N steps is L launches of N/L steps each (any N: no remainder
// steps), ping-ponging between the plan's two state buffers.  More steps per
// launch spread the launch's fixed cost (1.9 us between dependent kernels,
// the window's load and store) over more steps but widen the window's stale
// ends, and more points per lane need fewer workgroups but run longer per
// step, so the best pair depends on the field's size, on the 256 CUs it has to
// fill and on N.  The
// shapes' costs are those measured on MI355X (sw1d_wide.hpp), and wide_choose
// takes the cheapest pair.
//
// Measured against the swept diamonds at their best node width (both bitwise
// the oracle; point-updates/s of sustained runs, FP64):
//             2^10      2^14      2^16      2^18      2^20      2^21
//   KS     2.62e9    4.07e10   1.59e11   5.86e11   9.25e11   9.36e11   diamonds
//          5.10e9    7.9e10    2.28e11   6.4e11    1.08e12   1.18e12   wide
//   heat   1.02e10   1.58e11   6.2e11    2.23e12   4.95e12   5.1e12    diamonds
//          2.27e10   3.5e11    1.27e12   3.6e12    7.3e12    8.5e12    wide
//   Euler  3.5e8     5.5e9     2.1e10    4.3e10    5.5e10    5.8e10    diamonds
//          7.0e8     1.13e10   2.8e10    4.6e10    5.9e10    6.1e10    wide
// (Euler before, one wave per tile: 1.3e8, 2.1e9, 8.3e9, 2.3e10, 3.1e10, 3.2e10
// as trapezoids.)
// At 2^20 a KS launch of 64 steps takes 62 us: 53 us of FP64 issue at 4.04
// cycles per instruction (12.7% of it the window's overlap, 6.7% the halo
// lanes), 3% exchanges, the rest the launch.  FP32 KS on large fields is the one
// case the diamonds win (nodes of 512 points at 2^20: 1.33e12 against 1.12e12): FP32
// instructions of two waves co-issue, and the diamonds evaluate fewer points.  From
// which size, and at which node widths, takes_wide (sw1d_plan.hip) says.
// An Euler cell's step is some 460 instructions; at 2^20 a launch of 13 steps
// of 4 cells per lane takes 232 us, nine tenths of it FP64 issue, a quarter of
// which repeats neighbours' cells: the window's 928 cells lose 8 per step, and
// 234 registers per lane hold no more than 4 cells beside two waves per SIMD.

#include <cmath>

#include "sw1d_wide.hpp"

namespace sw1d {
namespace wide {
namespace {

template <typename T, int EQ, class S>
__global__ __launch_bounds__(S::NT) void k_wide(const T* __restrict__ in, T* __restrict__ out, int64_t n,
                                                int64_t wout, int steps, int ends, Coef<T, EQ> k)
{
    __shared__ __attribute__((aligned(16))) T lds[S::template lds<T>];
    const int64_t out0 = (int64_t)blockIdx.x * wout;
    const int count = (int)(n - out0 < wout ? n - out0 : wout);
    tile<T, EQ, S>(lds, in, out, n, n, out0, count, steps, ends, k);
}

template <typename T, int EQ, int I = 0>
hipError_t launch_shape(int shape, dim3 grid, const T* in, T* out, int64_t n, int64_t wout, int steps, int ends,
                        const Coefs& c, hipStream_t s)
{
    if constexpr (I < Table<EQ>::count) {
        if (shape != I) return launch_shape<T, EQ, I + 1>(shape, grid, in, out, n, wout, steps, ends, c, s);
        using S = TableShape<EQ, I>;
        hipLaunchKernelGGL((k_wide<T, EQ, S>), grid, dim3(S::NT), 0, s, in, out, n, wout, steps, ends,
                           (coef_of<T, EQ>(c)));
        return hipGetLastError();
    } else {
        return hipErrorInvalidValue;
    }
}

template <typename T>
hipError_t launch_prec(const WideLaunch& L, const Coefs& c, hipStream_t s)
{
    const int win = window(entries(L.eq)[L.shape]);
    const int64_t most = win - 2 * (int64_t)reach(L.eq) * L.steps;  // points a tile can store
    if (most < 1) return hipErrorInvalidValue;
    const int64_t tiles = (L.n + most - 1) / most, wout = (L.n + tiles - 1) / tiles;
    const dim3 grid((unsigned)((L.n + wout - 1) / wout));
    const int ends = L.bc == BC_MIRROR ? ENDS_MIRROR : L.bc == BC_DIRICHLET ? ENDS_FIXED : ENDS_PERIODIC;
    const T* in = static_cast<const T*>(L.in);
    T* out = static_cast<T*>(L.out);
    switch (L.eq) {
    case EQ_HEAT: return launch_shape<T, EQ_HEAT>(L.shape, grid, in, out, L.n, wout, L.steps, ends, c, s);
    case EQ_KS: return launch_shape<T, EQ_KS>(L.shape, grid, in, out, L.n, wout, L.steps, ends, c, s);
    case EQ_EULER: return launch_shape<T, EQ_EULER>(L.shape, grid, in, out, L.n, wout, L.steps, ends, c, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace
}  // namespace wide

hipError_t launch_wide(const WideLaunch& L, bool f64, const Coefs& c, hipStream_t s)
{
    return f64 ? wide::launch_prec<double>(L, c, s) : wide::launch_prec<float>(L, c, s);
}

WideChoice wide_choose(int eq, bool f64, int64_t n, int64_t nsteps, int cus)
{
    using namespace wide;
    WideChoice best;
    if (nsteps < 1) return best;
    const Entry* e = entries(eq);
    const int count = shapes(eq), r = reach(eq);
    const double points = (double)n, todo = (double)nsteps, units = cus > 0 ? cus : 256;
    for (int i = 0; i < count; ++i) {
        const Cost& c = f64 ? e[i].f64 : e[i].f32;
        const int win = window(e[i]);
        auto consider = [&](double stored) {  // most steps that leave a tile `stored` points
            double s = std::floor((win - stored) / (2 * r));
            if (!(s >= 1)) return;
            const double launches = std::ceil(todo / s);
            s = std::ceil(todo / launches);
            const double m = std::ceil(std::ceil(points / (win - 2 * r * s)) / units);
            const double us = launches * (c.t0 + (m - 1) * c.t2 + s * (c.c1 + (m - 1) * c.c2));
            if (best.launches == 0 || us < best.us) {
                best.shape = i;
                best.launches = (int64_t)launches;
                best.us = us;
            }
        };
        // a whole number of tiles on every CU, where the field has few tiles;
        // a share of the window, where it has many
        for (int m = 1; m <= 6; ++m) consider(std::ceil(points / (m * units)));
        for (double f : {.95, .9, .85, .8, .7, .6, .45, .3}) consider(f * win);
    }
    return best;
}

}  // namespace sw1d
