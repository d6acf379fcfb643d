// Device code of the workgroup-wide overlapped tile, shared by the single-plan
// kernels (sw1d_wide.hip) and the batched solve (sw1d_batch.hip).
//
// A workgroup of NW waves holds a window of consecutive points in VGPRs and
// advances it by any number of whole time steps; after s steps the points
// more than R s from the window's ends hold the classic scheme's values (R =
// points a value travels per step: 1 heat, 4 KS and Euler), and the tile
// stores those.  The wave is the unit that computes: lane l holds P
// consecutive points, neighbours cross lanes by DPP, and every lane updates
// every point it holds, so the steady loop has no mask, no select and no
// memory access: 12.5 instructions per KS point and stage, 12 of them FP64.
// Inside the workgroup the waves overlap by HL lanes on each side.  Those halo
// lanes go stale from the outside, and every K = HL P / R steps a wave takes
// its neighbours' values for them through LDS: a wave repeats 2 HL / 64 of its
// neighbours' work, and the workgroup repeats 2 R S / WIN of its neighbours'.
// An Euler wave updates cells of three values, and the waves that hold cell 0
// or n-1 run a variant with the Dirichlet ends' checks.
//
// Why a workgroup: the redundant share falls with the width of whatever
// shares its halo.  A wave alone (64 x 18 points) that advances KS by 16 steps
// repeats 11%, and a row of diamonds idles lanes outside its active set and
// pays a compare and two selects per point for it; four waves of 18 points
// per lane advance 48 steps for the same 11%.
#pragma once

#include "sw1d_euler.hpp"
#include "sw1d_internal.hpp"
#include "sw1d_lanes.hpp"

namespace sw1d {
namespace wide {

enum Ends : int { ENDS_PERIODIC = 0, ENDS_MIRROR = 1, ENDS_FIXED = 2 };

template <int EQ, int P_, int NW_, int HL_>
struct Shape {
    static constexpr int P = P_, NW = NW_, HL = HL_;
    static constexpr int NC = EQ == EQ_EULER ? 3 : 1;  // values per point between launches
    static constexpr int RS = EQ == EQ_HEAT ? 1 : 2;   // stencil radius of one stage
    static constexpr int R = EQ == EQ_HEAT ? 1 : 4;    // reach of one step
    static constexpr int NT = NW * kWave;
    static constexpr int STRIDE = (kWave - 2 * HL) * P;      // points a wave owns
    static constexpr int WIN = NW * STRIDE + 2 * HL * P;     // points of the window
    static constexpr int K = HL * P / R;                     // steps between exchanges
    static_assert(K >= 1 && 4 * HL <= kWave, "the halo lanes hold at least one step's reach");
    static constexpr int EDGE = NW * 2 * HL * NC * P;  // exchanged edges, in values
    // Lanes read and write the field themselves, 16 bytes at a time, where one
    // component's image after the other through LDS takes longer: Euler (4 cells
    // per lane: 8.6 us for launch, load and store against 5.5), heat up to eight
    // points per lane (5: 3.4 against 2.6 us; a field of 2^18 points, 4000 steps:
    // 361 -> 292 us in all) and FP32 KS up to five (3.0 against 2.1 us; 2^17, 1000
    // steps: 321 -> 288 us).  FP64 KS and wider FP32 tiles lose more in their
    // steps, whose registers the compiler then assigns worse (FP64, 4: 0.269
    // against 0.245 us per step; FP32, 6: 0.311 against 0.303), than they gain.
    template <typename T>
    static constexpr bool direct = P <= 2 || EQ == EQ_EULER || (EQ == EQ_HEAT ? P <= 8 : P <= 5 && sizeof(T) == 4);
    // LDS, in values: one component's window image, or the edges (two sets used
    // in turn, so one barrier per exchange is enough)
    template <typename T> static constexpr int lds = (!direct<T> && WIN > 2 * EDGE) ? WIN : 2 * EDGE;
};

// Field index of point g of the window, which may lie outside 0 .. n-1.
// Periodic: modulo n.  Mirror: reflected at both ends, T[-k] = T[k] (the
// insulated ends' T[-1] = T[1]); the stencil is symmetric, so the reflected
// points stay bitwise the mirror image and no end needs a check.  Fixed: the
// points outside are never used (the ends are pinned), any value will do.
__device__ __forceinline__ int64_t field_index(int64_t g, int64_t n, int ends, bool near)
{
    if (ends == ENDS_PERIODIC) {
        if (near) return g < 0 ? g + n : (g >= n ? g - n : g);
        const int32_t m = (int32_t)n;  // a window wider than the field: n is small
        const int32_t r = (int32_t)g % m;
        return r < 0 ? r + m : r;
    }
    if (ends == ENDS_MIRROR) {
        if (near) {
            g = g < 0 ? -g : g;
            return g >= n ? 2 * (n - 1) - g : g;
        }
        const int32_t m = 2 * ((int32_t)n - 1);
        int32_t r = (int32_t)g % m;
        r = r < 0 ? -r : r;
        return r < (int32_t)n ? r : m - r;
    }
    return g < 0 ? 0 : (g >= n ? n - 1 : g);
}

// 16-byte LDS copies of P values (d is 16-byte aligned when P is a multiple of
// 16 / sizeof(T); else the values go one by one)
template <typename T, int P>
__device__ __forceinline__ void put(T* d, const T (&v)[P])
{
    constexpr int V = 16 / sizeof(T);
    typedef T vec __attribute__((ext_vector_type(V)));
    if constexpr (P % V == 0) {
#pragma unroll
        for (int p = 0; p < P; p += V) {
            vec t;
#pragma unroll
            for (int q = 0; q < V; ++q) t[q] = v[p + q];
            *reinterpret_cast<vec*>(d + p) = t;
        }
    } else {
#pragma unroll
        for (int p = 0; p < P; ++p) d[p] = v[p];
    }
}
template <typename T, int P>
__device__ __forceinline__ void take(const T* d, T (&v)[P])
{
    constexpr int V = 16 / sizeof(T);
    typedef T vec __attribute__((ext_vector_type(V)));
    if constexpr (P % V == 0) {
#pragma unroll
        for (int p = 0; p < P; p += V) {
            const vec t = *reinterpret_cast<const vec*>(d + p);
#pragma unroll
            for (int q = 0; q < V; ++q) v[p + q] = t[q];
        }
    } else {
#pragma unroll
        for (int p = 0; p < P; ++p) v[p] = d[p];
    }
}

// P values at any element alignment, in 16-byte accesses where P allows them
// (a component starts at a multiple of n, which may be odd)
template <typename T, int P>
__device__ __forceinline__ void load_pts(const T* a, T (&v)[P])
{
    constexpr int V = P % (16 / sizeof(T)) == 0 ? 16 / sizeof(T) : (P % 2 == 0 ? 2 : 1);
    typedef T vec __attribute__((ext_vector_type(V), aligned(sizeof(T))));
#pragma unroll
    for (int p = 0; p < P; p += V) {
        const vec t = *reinterpret_cast<const vec*>(a + p);
#pragma unroll
        for (int q = 0; q < V; ++q) v[p + q] = t[q];
    }
}
template <typename T, int P>
__device__ __forceinline__ void store_pts(T* a, const T (&v)[P])
{
    constexpr int V = P % (16 / sizeof(T)) == 0 ? 16 / sizeof(T) : (P % 2 == 0 ? 2 : 1);
    typedef T vec __attribute__((ext_vector_type(V), aligned(sizeof(T))));
#pragma unroll
    for (int p = 0; p < P; p += V) {
        vec t;
#pragma unroll
        for (int q = 0; q < V; ++q) t[q] = v[p + q];
        *reinterpret_cast<vec*>(a + p) = t;
    }
}

// One Euler stage over the lane's P cells (Euler:307-389): dst = base + c
// flux(src), each interface once.  ENDS: this wave holds cell 0 or n-1, which
// take the Dirichlet states and drop the outermost pressure differences.
template <typename T, int P, bool ENDS>
__device__ __forceinline__ void euler_stage(const T (&src)[3][P], T (&dst)[3][P], const T (&base)[3][P],
                                            T (&hl)[3][2], T (&hr)[3][2], int c0, int cN, T c,
                                            const EulerCoef<T>& k)
{
    // c0 / cN: the lane's p of cell 0 / n-1
    auto drop0 = [&](int j) { return ENDS && j - 1 == c0; };
    auto drop2 = [&](int j) { return ENDS && j == cN; };
    eu_lane_stage<false, T, P>(src, hl, hr, k, drop0, drop2, [&](int p, const Q3<T>& f) {
        Q3<T> nv = eu_apply(Q3<T>{base[0][p], base[1][p], base[2][p]}, f, c);
        if (ENDS) {
            const bool l = p == c0, r = p == cN;
            nv = Q3<T>{l ? k.bl.x : nv.x, l ? k.bl.y : nv.y, l ? k.bl.z : nv.z};
            nv = Q3<T>{r ? k.br.x : nv.x, r ? k.br.y : nv.y, r ? k.br.z : nv.z};
        }
        dst[0][p] = nv.x;
        dst[1][p] = nv.y;
        dst[2][p] = nv.z;
    });
}

// An equation's own coefficients, a kernel argument: a launch takes longer with more
// bytes of arguments. With those of all three equations (more than 100 B in FP64) a plain
// launch took KS 2^10 4.3-4.9 us, heat 2^18 4.2-4.9 and heat 2^20 4.7-4.9; with its own
// 3.6-3.8, 3.4-3.8 and 4.1. FP64 Euler (104 B of its own) is as before, FP32 too.
template <typename T, int EQ> struct Coef;
template <typename T> struct Coef<T, EQ_HEAT> { T fo, fo2; };
template <typename T> struct Coef<T, EQ_KS> { KsCoef<T> ks; };
template <typename T> struct Coef<T, EQ_EULER> { EulerCoef<T> eu; };
template <typename T, int EQ>
inline Coef<T, EQ> coef_of(const Coefs& c)
{
    constexpr bool f64 = sizeof(T) == 8;
    if constexpr (EQ == EQ_HEAT) {
        if constexpr (f64) return {c.fo_d, c.fo2_d};
        else return {c.fo_f, c.fo2_f};
    } else if constexpr (EQ == EQ_KS) {
        if constexpr (f64) return {c.ks_d};
        else return {c.ks_f};
    } else {
        if constexpr (f64) return {c.eu_d};
        else return {c.eu_f};
    }
}

// k steps of the wave's points.  The lanes at the window's ends keep the
// neighbour they last had (carried registers): their points are stale anyway.
template <typename T, int EQ, class S>
struct Steps {
    static constexpr int P = S::P, NC = S::NC, RS = S::RS;
    T v[NC][P], q[NC][P];
    T hl[NC][RS], hr[NC][RS], gl[NC][RS], gr[NC][RS];

    __device__ __forceinline__ void start()
    {
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int i = 0; i < RS; ++i) hl[c][i] = hr[c][i] = gl[c][i] = gr[c][i] = v[c][0];
    }
    __device__ __forceinline__ void heat(const T (&s)[P], T (&d)[P], T (&a)[1], T (&b)[1], const Coef<T, EQ>& k)
    {
        T e[P + 2];
        gather_carry<T, P, 1>(s, a, b, e);
#pragma unroll
        for (int p = 0; p < P; ++p) d[p] = heat_ftcs(e[p], e[p + 1], e[p + 2], k.fo, k.fo2);
    }
    template <bool ENDS>
    __device__ __forceinline__ void run(int steps, const Coef<T, EQ>& k, int c0, int cN)
    {
        if constexpr (EQ == EQ_HEAT) {
            if (steps & 1) {
                heat(v[0], q[0], hl[0], hr[0], k);
#pragma unroll
                for (int p = 0; p < P; ++p) v[0][p] = q[0][p];
            }
            for (int s = steps >> 1; s > 0; --s) {
                heat(v[0], q[0], hl[0], hr[0], k);
                heat(q[0], v[0], gl[0], gr[0], k);
            }
        } else if constexpr (EQ == EQ_KS) {
            for (int s = steps; s > 0; --s) {
                {
                    T e[P + 4];
                    gather_carry<T, P, 2>(v[0], hl[0], hr[0], e);
#pragma unroll
                    for (int p = 0; p < P; ++p)
                        q[0][p] = ks_predict(e[p], e[p + 1], e[p + 2], e[p + 3], e[p + 4], k.ks);
                }
                {
                    T e[P + 4];
                    gather_carry<T, P, 2>(q[0], gl[0], gr[0], e);
#pragma unroll
                    for (int p = 0; p < P; ++p)
                        v[0][p] = ks_correct(v[0][p], e[p], e[p + 1], e[p + 2], e[p + 3], e[p + 4], k.ks);
                }
            }
        } else {
            const T ca = T(0.25) * k.eu.dtdx, cb = T(0.5) * k.eu.dtdx;
            for (int s = steps; s > 0; --s) {
                euler_stage<T, P, ENDS>(v, q, v, hl, hr, c0, cN, ca, k.eu);  // predictor
                euler_stage<T, P, ENDS>(q, v, v, gl, gr, c0, cN, cb, k.eu);  // corrector
            }
        }
    }
};

// One tile: out[out0 .. out0 + count) after `steps` steps from the field `in`
// of n points (component stride cs in both).  The window starts R steps
// before out0; lds holds Shape::lds<T> values.
template <typename T, int EQ, class S>
__device__ __forceinline__ void tile(T* lds, const T* __restrict__ in, T* __restrict__ out, int64_t n, int64_t cs,
                                     int64_t out0, int count, int steps, int ends,
                                     const Coef<T, EQ>& k)
{
    constexpr int P = S::P, NW = S::NW, HL = S::HL, NC = S::NC, NT = S::NT, WIN = S::WIN;
    constexpr int NL = (WIN + NT - 1) / NT;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), w = tid >> 6;
    const int halo = S::R * steps;
    const int64_t win = out0 - halo;
    const int x0 = w * S::STRIDE + lane * P;  // window position of the lane's first point
    const bool inside = win >= 0 && win + WIN <= n;
    const bool near = win >= -(n - 1) && win + WIN <= 2 * n - 1;
    Steps<T, EQ, S> st;
    if constexpr (S::template direct<T>) {
        if (inside) {
#pragma unroll
            for (int c = 0; c < NC; ++c) load_pts<T, P>(in + c * cs + win + x0, st.v[c]);
        } else {
#pragma unroll
            for (int p = 0; p < P; ++p) {
                const int64_t g = field_index(win + x0 + p, n, ends, near);
#pragma unroll
                for (int c = 0; c < NC; ++c) st.v[c][p] = in[c * cs + g];
            }
        }
    } else {
        // coalesced through the LDS image, every load of a component in flight
        // at once (also where the window wraps: one slow tile would hold up
        // the whole launch)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            T r[NL];
            if (inside) {
                const T* a = in + c * cs + win;
#pragma unroll
                for (int j = 0; j < NL; ++j)
                    if (tid + j * NT < WIN) r[j] = a[tid + j * NT];
            } else {
#pragma unroll
                for (int j = 0; j < NL; ++j)
                    if (tid + j * NT < WIN) r[j] = in[c * cs + field_index(win + tid + j * NT, n, ends, near)];
            }
            if (c > 0) __syncthreads();  // the previous component's image has been read
#pragma unroll
            for (int j = 0; j < NL; ++j)
                if (tid + j * NT < WIN) lds[tid + j * NT] = r[j];
            __syncthreads();
#pragma unroll
            for (int p = 0; p < P; ++p) st.v[c][p] = lds[x0 + p];
        }
        __syncthreads();
    }
    st.start();
    // Euler's Dirichlet cells 0 and n-1: the lane's p of each where one of its
    // interfaces touches it (c0 = -1 and cN = P: the neighbour lane's cell)
    int c0 = -9, cN = -9;
    bool fixed = false;
    if constexpr (EQ == EQ_EULER) {
        const int64_t g = win + x0;
        if (g <= 1 && g > -P) c0 = (int)-g;
        if (n - 1 - g >= 0 && n - 1 - g <= P) cN = (int)(n - 1 - g);
        fixed = __builtin_amdgcn_ballot_w64(c0 != -9 || cN != -9) != 0;
    }

    const bool left = lane < 2 * HL;
    const bool wr = (lane >= HL && left) || (lane >= kWave - 2 * HL && lane < kWave - HL);
    const bool rd = (lane < HL && w > 0) || (lane >= kWave - HL && w < NW - 1);
    // edge slot (wave, side, lane within the edge): a wave writes its own two
    // edges and reads the facing ones of its neighbours
    const int wslot = left ? (2 * w) * HL + lane - HL : (2 * w + 1) * HL + lane - (kWave - 2 * HL);
    const int rslot = left ? (2 * w - 1) * HL + lane : (2 * w + 2) * HL + lane - (kWave - HL);
    int todo = steps, set = 0;
    for (;;) {
        const int s = NW == 1 || todo < S::K ? todo : S::K;
        todo -= s;
        if constexpr (EQ == EQ_EULER) {
            if (fixed)
                st.template run<true>(s, k, c0, cN);
            else
                st.template run<false>(s, k, c0, cN);
        } else {
            st.template run<false>(s, k, c0, cN);
        }
        if (todo <= 0) break;
        T* e = lds + set;
        set = S::EDGE - set;
        if (wr) {
#pragma unroll
            for (int c = 0; c < NC; ++c) put<T, P>(e + (wslot * NC + c) * P, st.v[c]);
        }
        __syncthreads();
        if (rd) {
#pragma unroll
            for (int c = 0; c < NC; ++c) take<T, P>(e + (rslot * NC + c) * P, st.v[c]);
        }
    }

    const bool own = (lane >= HL || w == 0) && (lane < kWave - HL || w == NW - 1);
    if constexpr (S::template direct<T>) {
        const int i0 = x0 - halo;
        if (own && i0 >= 0 && i0 + P <= count) {
#pragma unroll
            for (int c = 0; c < NC; ++c) store_pts<T, P>(out + c * cs + out0 + i0, st.v[c]);
        } else if (own) {
#pragma unroll
            for (int p = 0; p < P; ++p) {
                if (i0 + p >= 0 && i0 + p < count) {
#pragma unroll
                    for (int c = 0; c < NC; ++c) out[c * cs + out0 + i0 + p] = st.v[c][p];
                }
            }
        }
    } else {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            __syncthreads();  // the last edges, or the previous component, have been read
            if (own) {
#pragma unroll
                for (int p = 0; p < P; ++p) lds[x0 + p] = st.v[c][p];
            }
            __syncthreads();
            T r[NL];
#pragma unroll
            for (int j = 0; j < NL; ++j)
                if (tid + j * NT < count) r[j] = lds[halo + tid + j * NT];
            T* o = out + c * cs + out0;
#pragma unroll
            for (int j = 0; j < NL; ++j)
                if (tid + j * NT < count) o[tid + j * NT] = r[j];
        }
    }
}

// ---------------------------------------------------------------- shapes ---
// A shape and its measured cost, in microseconds: a launch of s steps whose
// CUs each take m workgroups costs
//   t0 + (m - 1) t2 + s (c1 + (m - 1) c2)
// (t0: launch, load, store; c1: one workgroup alone on its CU, bound by issue
// from about six points per lane and by latency below; c2: each further one).
struct Cost { float t0, t2, c1, c2; };
struct Entry { int P, HL; Cost f64, f32; };

inline constexpr int kWaves = 4;  // one wave per SIMD: P sets the window
// Halo lanes: an exchange every HL P / R steps, 5-9 for KS, 16-42 for heat and 2-5
// for Euler, whose steps are ten times as long
inline constexpr Entry kKs[] = {
    {2, 10, {2.3f, .06f, .151f, .101f}, {2.1f, .02f, .143f, .085f}},
    {4, 6, {3.0f, .6f, .248f, .173f}, {2.35f, .3f, .2245f, .1535f}},
    {5, 4, {3.2f, .45f, .319f, .217f}, {2.15f, .3f, .300f, .188f}},
    {6, 4, {3.6f, .4f, .318f, .268f}, {3.3f, .25f, .301f, .226f}},
    {8, 4, {4.7f, .4f, .383f, .36f}, {3.7f, .2f, .377f, .296f}},
    {10, 2, {4.8f, .4f, .508f, .46f}, {4.2f, .35f, .469f, .374f}},
    {12, 2, {5.6f, .6f, .590f, .56f}, {4.9f, .35f, .540f, .43f}},
    {14, 2, {6.0f, .5f, .634f, .66f}, {5.2f, .35f, .619f, .44f}},
    {16, 2, {7.0f, .7f, .709f, .75f}, {5.7f, .3f, .698f, .56f}},
    {19, 2, {8.5f, .9f, .834f, .87f}, {6.4f, .25f, .816f, .68f}},
};
inline constexpr Entry kHeat[] = {
    {2, 8, {2.1f, .18f, .0350f, .0151f}, {2.1f, .08f, .0299f, .0110f}},
    {3, 8, {2.2f, .35f, .0420f, .0197f}, {2.35f, .1f, .0358f, .0163f}},
    {4, 6, {2.35f, .45f, .0432f, .0245f}, {2.2f, .2f, .0410f, .0200f}},
    {5, 4, {2.6f, .45f, .0503f, .0290f}, {2.35f, .2f, .0447f, .0256f}},
    {7, 4, {3.0f, .6f, .0610f, .0355f}, {2.7f, .3f, .0542f, .0325f}},
    {9, 4, {4.1f, .5f, .0673f, .0462f}, {3.8f, .3f, .0625f, .0423f}},
    {12, 2, {4.8f, .6f, .0875f, .0622f}, {4.3f, .37f, .0819f, .0539f}},
    {15, 2, {5.6f, .7f, .106f, .0770f}, {5.0f, .3f, .0956f, .0623f}},
    {19, 2, {7.0f, .7f, .1203f, .0970f}, {5.8f, .3f, .1128f, .0811f}},
    {21, 2, {7.4f, .9f, .1305f, .1066f}, {6.2f, .25f, .1226f, .0892f}},
};

inline constexpr Entry kEuler[] = {
    {1, 16, {2.2f, .0f, 1.29f, .85f}, {2.0f, .1f, 1.09f, .56f}},
    {1, 8, {1.75f, .4f, 1.37f, .82f}, {1.8f, .2f, 1.16f, .56f}},
    {2, 8, {2.3f, .9f, 2.30f, 1.60f}, {2.1f, .15f, 2.00f, 1.13f}},
    {2, 4, {2.7f, .9f, 2.35f, 1.58f}, {2.4f, .3f, 2.08f, 1.12f}},
    {3, 4, {4.3f, 1.6f, 3.34f, 2.41f}, {2.7f, .9f, 2.87f, 1.68f}},
    {4, 4, {5.5f, 2.2f, 4.35f, 3.10f}, {3.7f, .9f, 3.78f, 2.25f}},
    {5, 4, {9.4f, 2.5f, 5.27f, 5.15f}, {4.2f, 1.5f, 4.64f, 2.82f}},
    {6, 2, {8.3f, 4.0f, 6.63f, 6.20f}, {3.5f, 2.0f, 5.65f, 3.20f}},
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
template <> struct Table<EQ_EULER> {
    static constexpr const Entry* e = kEuler;
    static constexpr int count = sizeof(kEuler) / sizeof(Entry);
};
template <int EQ, int I> using TableShape = Shape<EQ, Table<EQ>::e[I].P, kWaves, Table<EQ>::e[I].HL>;
inline const Entry* entries(int eq) { return eq == EQ_HEAT ? kHeat : eq == EQ_KS ? kKs : kEuler; }
inline int shapes(int eq)
{
    return eq == EQ_HEAT ? Table<EQ_HEAT>::count : eq == EQ_KS ? Table<EQ_KS>::count : Table<EQ_EULER>::count;
}

}  // namespace wide
}  // namespace sw1d
