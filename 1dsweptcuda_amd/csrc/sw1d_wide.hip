// Workgroup-wide overlapped tiles (sw1d_wide.hpp) for single heat and KS plans:
// the kernels, and the choice of a tile shape and of the steps per launch.
//
// An advance of N steps is L launches of N/L steps each (any N: no remainder
// steps), ping-ponging between the plan's two state buffers.  More steps per
// launch spread the launch's fixed cost (1.9 us between dependent kernels,
// the window's load and store) over more steps but widen the window's stale
// ends, and more points per lane need fewer workgroups but run longer per
// step, so the best pair depends on the field's size, on the 256 CUs it has to
// fill and on N.  kShapes holds each shape's cost as measured on MI355X and
// wide_choose takes the cheapest pair.
//
// Measured against the swept diamonds at their best node width (both bitwise
// the oracle; point-updates/s of sustained runs, FP64):
//             2^10      2^14      2^16      2^18      2^20      2^21
//   KS     2.62e9    4.07e10   1.59e11   5.86e11   9.25e11   9.36e11   diamonds
//          5.10e9    7.9e10    2.28e11   6.4e11    1.08e12   1.18e12   wide
//   heat   1.02e10   1.58e11   6.2e11    2.23e12   4.95e12   5.1e12    diamonds
//          2.18e10   3.35e11   1.14e12   3.4e12    7.1e12    8.5e12    wide
// At 2^20 a KS launch of 64 steps takes 62 us: 53 us of FP64 issue at 4.04
// cycles per instruction (12.7% of it the window's overlap, 6.7% the halo
// lanes), 3% exchanges, the rest the launch.  FP32 KS at 2^19 and more is the
// one case the diamonds win (1.32e12 against 1.14e12 at 2^20): FP32
// instructions of two waves co-issue, and the diamonds evaluate fewer points.

#include <cmath>

#include "sw1d_wide.hpp"

namespace sw1d {
namespace wide {
namespace {

template <typename T, int EQ, class S>
__global__ __launch_bounds__(S::NT) void k_wide(const T* __restrict__ in, T* __restrict__ out, int64_t n,
                                                int64_t wout, int steps, int ends, Coef<T> k)
{
    __shared__ __attribute__((aligned(16))) T lds[S::LDS];
    const int64_t out0 = (int64_t)blockIdx.x * wout;
    const int count = (int)(n - out0 < wout ? n - out0 : wout);
    tile<T, EQ, S>(lds, in, out, n, n, out0, count, steps, ends, k);
}

// A shape and its measured cost, in microseconds: a launch of s steps whose
// CUs each take m workgroups costs
//   t0 + (m - 1) t2 + s (c1 + (m - 1) c2)
// (t0: launch, load, store; c1: one workgroup alone on its CU, bound by issue
// from about six points per lane and by latency below; c2: each further one).
struct Cost { float t0, t2, c1, c2; };
struct Entry { int P, HL; Cost f64, f32; };

constexpr int kWaves = 4;  // one wave per SIMD: P sets the window
// Halo lanes: an exchange every HL P / R steps, 5-9 for KS and 16-42 for heat
constexpr Entry kKs[] = {
    {2, 10, {2.3f, .06f, .151f, .101f}, {2.1f, .02f, .143f, .085f}},
    {4, 6, {3.0f, .6f, .248f, .173f}, {2.8f, .35f, .224f, .153f}},
    {5, 4, {3.2f, .45f, .319f, .217f}, {3.0f, .2f, .301f, .193f}},
    {6, 4, {3.6f, .4f, .318f, .268f}, {3.3f, .25f, .301f, .226f}},
    {8, 4, {4.7f, .4f, .383f, .36f}, {3.7f, .2f, .377f, .296f}},
    {10, 2, {4.8f, .4f, .508f, .46f}, {4.2f, .35f, .469f, .374f}},
    {12, 2, {5.6f, .6f, .590f, .56f}, {4.9f, .35f, .540f, .43f}},
    {14, 2, {6.0f, .5f, .634f, .66f}, {5.2f, .35f, .619f, .44f}},
    {16, 2, {7.0f, .7f, .709f, .75f}, {5.7f, .3f, .698f, .56f}},
    {19, 2, {8.5f, .9f, .834f, .87f}, {6.4f, .25f, .816f, .68f}},
};
constexpr Entry kHeat[] = {
    {2, 8, {2.1f, .18f, .0371f, .0151f}, {2.1f, .08f, .0299f, .0110f}},
    {3, 8, {2.7f, .38f, .0407f, .0193f}, {2.7f, .15f, .0348f, .0162f}},
    {4, 6, {3.1f, .5f, .0446f, .0247f}, {2.9f, .2f, .0393f, .0199f}},
    {5, 4, {3.3f, .4f, .0511f, .0292f}, {3.0f, .17f, .0482f, .0258f}},
    {7, 4, {3.3f, .45f, .0621f, .0379f}, {3.3f, .25f, .0650f, .0330f}},
    {9, 4, {4.1f, .5f, .0673f, .0462f}, {3.8f, .3f, .0625f, .0423f}},
    {12, 2, {4.8f, .6f, .0875f, .0622f}, {4.3f, .37f, .0819f, .0539f}},
    {15, 2, {5.6f, .7f, .106f, .0770f}, {5.0f, .3f, .0956f, .0623f}},
    {19, 2, {7.0f, .7f, .1203f, .0970f}, {5.8f, .3f, .1128f, .0811f}},
    {21, 2, {7.4f, .9f, .1305f, .1066f}, {6.2f, .25f, .1226f, .0892f}},
};

inline int reach(int eq) { return eq == EQ_HEAT ? 1 : 4; }
inline int window(const Entry& e) { return kWaves * (kWave - 2 * e.HL) * e.P + 2 * e.HL * e.P; }

template <int EQ> struct Table;
template <> struct Table<EQ_HEAT> {
    static constexpr const Entry* e = kHeat;
    static constexpr int count = sizeof(kHeat) / sizeof(Entry);
};
template <> struct Table<EQ_KS> {
    static constexpr const Entry* e = kKs;
    static constexpr int count = sizeof(kKs) / sizeof(Entry);
};

template <typename T, int EQ, int I = 0>
hipError_t launch_shape(int shape, dim3 grid, const T* in, T* out, int64_t n, int64_t wout, int steps, int ends,
                        const Coef<T>& k, hipStream_t s)
{
    if constexpr (I < Table<EQ>::count) {
        if (shape != I) return launch_shape<T, EQ, I + 1>(shape, grid, in, out, n, wout, steps, ends, k, s);
        using S = Shape<EQ, Table<EQ>::e[I].P, kWaves, Table<EQ>::e[I].HL>;
        hipLaunchKernelGGL((k_wide<T, EQ, S>), grid, dim3(S::NT), 0, s, in, out, n, wout, steps, ends, k);
        return hipGetLastError();
    } else {
        return hipErrorInvalidValue;
    }
}

template <typename T>
hipError_t launch_prec(const WideLaunch& L, const Coefs& c, hipStream_t s)
{
    Coef<T> k{};
    if constexpr (sizeof(T) == 8) {
        k.fo = c.fo_d; k.fo2 = c.fo2_d; k.ks = c.ks_d;
    } else {
        k.fo = c.fo_f; k.fo2 = c.fo2_f; k.ks = c.ks_f;
    }
    const int win = window(L.eq == EQ_HEAT ? kHeat[L.shape] : kKs[L.shape]);
    const int64_t most = win - 2 * (int64_t)reach(L.eq) * L.steps;  // points a tile can store
    if (most < 1) return hipErrorInvalidValue;
    const int64_t tiles = (L.n + most - 1) / most, wout = (L.n + tiles - 1) / tiles;
    const dim3 grid((unsigned)((L.n + wout - 1) / wout));
    const int ends = L.bc == BC_MIRROR ? ENDS_MIRROR : ENDS_PERIODIC;
    const T* in = static_cast<const T*>(L.in);
    T* out = static_cast<T*>(L.out);
    return L.eq == EQ_HEAT ? launch_shape<T, EQ_HEAT>(L.shape, grid, in, out, L.n, wout, L.steps, ends, k, s)
                           : launch_shape<T, EQ_KS>(L.shape, grid, in, out, L.n, wout, L.steps, ends, k, s);
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
    const Entry* e = eq == EQ_HEAT ? kHeat : kKs;
    const int count = eq == EQ_HEAT ? Table<EQ_HEAT>::count : Table<EQ_KS>::count;
    const int r = reach(eq);
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
