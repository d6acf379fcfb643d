// One classic time step per launch, both Runge-Kutta stages in it.
//
// Each wave64 advances 64 P consecutive points by one step in VGPRs with the
// stages of the wide tiles (sw1d_wide.hpp) and stores those at least R points
// from its ends: the halo lanes' points are also the neighbouring wave's.  No
// LDS and no barrier, so the waves of a workgroup are independent; a point is
// read and written once per step, where a launch per stage moved KS's u and
// u_half (Euler's six values) five times and paid the 1.9 us between
// dependent kernels twice.  Heat's step is one stage.
//
// Replayed from a graph a small step is bound by that gap, one of 2^20 heat or
// KS points by the state's way through the caches, a large Euler step by FP64
// issue.  us per step, FP64, a launch per stage -> this kernel:
//   KS 2^14 3.92 -> 2.04, 2^20 7.6 -> 4.1, 2^22 26.5 -> 11.6;
//   Euler 2^14 5.7 -> 3.1, 2^20 37 -> 15.7 (Sod) to 20.9 (cells that all differ);
//   heat 2^20 4.5 -> 3.6

#include "sw1d_wide.hpp"

namespace sw1d {
namespace wide {
namespace {

constexpr int kStepBlock = 256;
// halo lanes on each side: one step's reach
template <int EQ, int P> constexpr int kHalo = ((EQ == EQ_HEAT ? 1 : 4) + P - 1) / P;

template <typename T, int EQ, int P>
__global__ __launch_bounds__(kStepBlock) void k_step(const T* __restrict__ in, T* __restrict__ out, int64_t n,
                                                     int ends, Coef<T, EQ> k)
{
    constexpr int HL = kHalo<EQ, P>;
    using S = Shape<EQ, P, 1, HL>;
    constexpr int NC = S::NC, OWN = (kWave - 2 * HL) * P;
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t first = ((int64_t)blockIdx.x * (kStepBlock / kWave) + (threadIdx.x >> 6)) * OWN;
    if (first >= n) return;  // the whole wave
    const int64_t win = first - HL * P, x = win + lane * P;
    Steps<T, EQ, S> st;
    if (win >= 0 && win + kWave * P <= n) {
#pragma unroll
        for (int c = 0; c < NC; ++c) load_pts<T, P>(in + c * n + x, st.v[c]);
    } else {
        const bool near = win >= -(n - 1) && win + kWave * P <= 2 * n - 1;
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const int64_t g = field_index(x + p, n, ends, near);
#pragma unroll
            for (int c = 0; c < NC; ++c) st.v[c][p] = in[c * n + g];
        }
    }
    st.start();
    if constexpr (EQ == EQ_EULER) {
        int c0 = -9, cN = -9;
        // as in tile(): the lane's p of the Dirichlet cells 0 and n-1
        if (x <= 1 && x > -P) c0 = (int)-x;
        if (n - 1 - x >= 0 && n - 1 - x <= P) cN = (int)(n - 1 - x);
        if (__builtin_amdgcn_ballot_w64(c0 != -9 || cN != -9) != 0)
            st.template run<true>(1, k, c0, cN);
        else
            st.template run<false>(1, k, c0, cN);
    } else {
        st.template run<false>(1, k, 0, 0);
    }
    if (lane < HL || lane >= kWave - HL) return;
    if (x + P <= n) {
#pragma unroll
        for (int c = 0; c < NC; ++c) store_pts<T, P>(out + c * n + x, st.v[c]);
    } else {
#pragma unroll
        for (int p = 0; p < P; ++p)
            if (x + p < n) {
#pragma unroll
                for (int c = 0; c < NC; ++c) out[c * n + x + p] = st.v[c][p];
            }
    }
}

// A heat step of a small field: one point per thread, the neighbours loaded
// too (the three loads are in flight together, nothing follows but the update).
// The kind of ends is a template argument: chosen at run time it became branches,
// each waiting for an argument load of its own (2^17 points, FP64: 2.18 against
// 2.16 us per step).
template <typename T, bool PERIODIC>
__global__ __launch_bounds__(kStepBlock) void k_heat_point(const T* __restrict__ in, T* __restrict__ out, int64_t n,
                                                           T fo, T fo2)
{
    const int64_t i = (int64_t)blockIdx.x * kStepBlock + threadIdx.x;
    if (i >= n) return;
    const int64_t l = i == 0 ? (PERIODIC ? n - 1 : 1) : i - 1, r = i == n - 1 ? (PERIODIC ? 0 : n - 2) : i + 1;
    out[i] = heat_ftcs(in[l], in[i], in[r], fo, fo2);
}

template <typename T, int EQ, int P>
hipError_t step_points(int64_t n, int ends, const T* in, T* out, const Coefs& c, hipStream_t s)
{
    constexpr int64_t own = (kWave - 2 * kHalo<EQ, P>) * P * (kStepBlock / kWave);
    hipLaunchKernelGGL((k_step<T, EQ, P>), dim3((unsigned)((n + own - 1) / own)), dim3(kStepBlock), 0, s, in, out, n,
                       ends, (coef_of<T, EQ>(c)));
    return hipGetLastError();
}

// Points per lane.  KS: one while that gives a SIMD no more than one wave (a
// step is then as long as a wave lives: 2^10 1.9 us against 2.0 in FP64 and
// 2.1 in FP32), else 16 bytes, the widest load (2^20: 4.1 against 4.7 us in
// FP64, 3.2 against 3.9 in FP32).  Heat: a point per thread up to two waves
// per SIMD in FP64 (150001 points: 2.20 us with 16 bytes against 2.26) and seven in
// FP32 (2^18: 2.13 against 2.25; 400001: 2.25 against 2.38; 2^19: 2.37 both), else
// 16 bytes (2^20: 3.65 against 4.55, 2.75 against 3.38); means over plans at 14
// places in memory, which alone make 5% of a step.  Euler: one up to eight
// waves per SIMD (2^18: 7.9 against 8.7 us), where latency no longer counts
// two, whose halo repeats 4 of 64 lanes instead of 8 (2^20, at the time: 22.4
// against 23.9).
template <typename T>
hipError_t step_prec(int eq, int bc, int64_t n, int simds, const void* in, void* out, const Coefs& c, hipStream_t s)
{
    constexpr int V = 16 / sizeof(T);
    const T* a = static_cast<const T*>(in);
    T* b = static_cast<T*>(out);
    const int64_t waves = n / 56;  // of KS and Euler at one point per lane
    if (eq == EQ_HEAT) {
        const bool periodic = bc != BC_MIRROR;
        if (n > (sizeof(T) == 8 ? 2 : 7) * kWave * (int64_t)simds)
            return step_points<T, EQ_HEAT, V>(n, periodic ? ENDS_PERIODIC : ENDS_MIRROR, a, b, c, s);
        const dim3 grid((unsigned)((n + kStepBlock - 1) / kStepBlock));
        const Coef<T, EQ_HEAT> k = coef_of<T, EQ_HEAT>(c);
        if (periodic)
            hipLaunchKernelGGL((k_heat_point<T, true>), grid, dim3(kStepBlock), 0, s, a, b, n, k.fo, k.fo2);
        else
            hipLaunchKernelGGL((k_heat_point<T, false>), grid, dim3(kStepBlock), 0, s, a, b, n, k.fo, k.fo2);
        return hipGetLastError();
    }
    if (eq == EQ_KS)
        return waves <= simds ? step_points<T, EQ_KS, 1>(n, ENDS_PERIODIC, a, b, c, s)
                              : step_points<T, EQ_KS, V>(n, ENDS_PERIODIC, a, b, c, s);
    if (eq == EQ_EULER)
        return waves <= 8 * (int64_t)simds ? step_points<T, EQ_EULER, 1>(n, ENDS_FIXED, a, b, c, s)
                                           : step_points<T, EQ_EULER, 2>(n, ENDS_FIXED, a, b, c, s);
    return hipErrorInvalidValue;
}

}  // namespace
}  // namespace wide

hipError_t launch_step(int eq, int bc, bool f64, int64_t n, int simds, const void* in, void* out, const Coefs& c,
                       hipStream_t s)
{
    return f64 ? wide::step_prec<double>(eq, bc, n, simds, in, out, c, s)
               : wide::step_prec<float>(eq, bc, n, simds, in, out, c, s);
}

}  // namespace sw1d
