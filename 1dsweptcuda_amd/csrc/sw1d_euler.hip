// gfx950 kernels of the Euler equations: the swept tiles and the classic
// stages.  The tile scheme is that of sw1d_kernels.hip (one wave per node,
// staggered levels, masked active sets, centred regions).

#include "sw1d_euler.hpp"
#include "sw1d_nodes.hpp"

namespace sw1d {
namespace {

// ---------------------------------------------------------- Euler tiles ---
// Components 0..2 are the conserved values (rho, rho*u, E), 3..5 their
// predictor.  EulerRegion holds PC cells per lane of the middle 64*PC cells
// of a node (all of it when PC = P).
template <typename T, int PC>
struct EulerRegion {
    T q[6][PC];
    T hl[6][2], hr[6][2];
    int d[PC];
    bool g0, gN;  // this lane's first / last cell is global cell 0 / n-1
    // one cell per lane: the lane's cell is global cell 1 / n-2 (with two or
    // more per lane, cells 0 and 1, and n-2 and n-1, share a lane)
    bool g1 = false, gNm1 = false;

    // src = 0: predictor from the conserved values (Euler:307-350);
    // src = 3: corrector from the predictor values (Euler:353-389, :420).
    // FULL: the stage's active set is the whole region, its end cells included
    // (the last corrector of a region's down phase, thr = 64 PC - 1); at every
    // other stage the two outermost cells on each side keep their values, and
    // the interfaces that only they use are not evaluated.
    template <int src, bool FULL>
    __device__ __forceinline__ void stage(int thr, const EulerCoef<T>& k)
    {
        constexpr int dst = 3 - src;
        const T c = src == 0 ? T(0.25) * k.dtdx : T(0.5) * k.dtdx;
        // the interface left of global cell 1 drops pdiff(-1,0), the one right
        // of cell n-2 drops pdiff(n-1,n) (the flags of Euler:405, :424)
        auto drop0 = [&](int j) { return (j == 1 && g0) || (PC == 1 && j == 0 && g1); };
        auto drop2 = [&](int j) { return (j == PC - 1 && gN) || (PC == 1 && j == 1 && gNm1); };
        eu_lane_stage<FULL, T, PC>(&q[src], &hl[src], &hr[src], k, drop0, drop2, [&](int p, const Q3<T>& f) {
            Q3<T> nv = eu_apply(Q3<T>{q[0][p], q[1][p], q[2][p]}, f, c);
            // ghost cells 0 and n-1 hold the Dirichlet states (Euler:405-425)
            if (p == 0 && g0) nv = k.bl;
            if (p == PC - 1 && gN) nv = k.br;
            const bool act = d[p] <= thr;
            q[dst + 0][p] = act ? nv.x : q[dst + 0][p];
            q[dst + 1][p] = act ? nv.y : q[dst + 1][p];
            q[dst + 2][p] = act ? nv.z : q[dst + 2][p];
        });
    }
    // down pairs s = s0, s0+2, .. s1; the last corrector's active set is the
    // whole region
    __device__ __forceinline__ void down(int s0, int s1, const EulerCoef<T>& k)
    {
        for (int s = s0; s <= s1; s += 2) {
            stage<0, false>(4 * s - 1, k);
            if (s < s1)
                stage<3, false>(4 * s + 3, k);
            else
                stage<3, true>(4 * s + 3, k);
        }
    }
    __device__ __forceinline__ void up(int W, int m0, int m1, const EulerCoef<T>& k)
    {
        for (int m = m0; m <= m1; m += 2) { stage<0, false>(W - 1 - 4 * m, k); stage<3, false>(W - 5 - 4 * m, k); }
    }
    __device__ __forceinline__ void place(int W, int x0, int64_t base, int64_t n)
    {
#pragma unroll
        for (int p = 0; p < PC; ++p) d[p] = abs(2 * (x0 + p) - (W - 1));
        int64_t gi = base + x0;
        gi = gi >= n ? gi - n : gi;
        int64_t gl = gi + PC - 1;
        gl = gl >= n ? gl - n : gl;
        g0 = gi == 0;
        gN = gl == n - 1;
        if (PC == 1) {
            g1 = gi == 1;
            gNm1 = gl == n - 2;
        }
    }
    // The region is the middle 64*PC cells of a node of W cells (all of it
    // when PC = W/64): lane l holds node-local x0 = W/2 - 32 PC + l PC ..
    // x0 + PC - 1, and the halo is the two cells beyond each end.
    template <int W>
    static constexpr int xs() { return W / 2 - 32 * PC; }
    // every component and the halo from the state arrays (node base `base`)
    template <int W>
    __device__ __forceinline__ void load_global(const T* in, int64_t n, int64_t base, int lane)
    {
        const int x0 = xs<W>() + lane * PC;
#pragma unroll
        for (int c = 0; c < 6; ++c) {
#pragma unroll
            for (int p = 0; p < PC; ++p) q[c][p] = in[c * n + wrap(base + x0 + p, n)];
        }
        halo_global<W>(in, n, base);
    }
    template <int W>
    __device__ __forceinline__ void halo_global(const T* in, int64_t n, int64_t base)
    {
#pragma unroll
        for (int c = 0; c < 6; ++c) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                hl[c][i] = in[c * n + wrap(base + xs<W>() - 1 - i, n)];
                hr[c][i] = in[c * n + wrap(base + xs<W>() + 64 * PC + i, n)];
            }
        }
    }
    // Components C0 .. C0+2 to / from a three-component node image (component
    // c at img + (c - C0) W, node-local cell order).
    template <int W, int C0>
    __device__ __forceinline__ void save_half(T* img, int lane) const
    {
        const int x0 = xs<W>() + lane * PC;
#pragma unroll
        for (int c = C0; c < C0 + 3; ++c)
#pragma unroll
            for (int p = 0; p < PC; ++p) img[(c - C0) * W + x0 + p] = q[c][p];
    }
    template <int W, int C0>
    __device__ __forceinline__ void load_half(const T* img, int lane)
    {
        const int x0 = xs<W>() + lane * PC;
#pragma unroll
        for (int c = C0; c < C0 + 3; ++c)
#pragma unroll
            for (int p = 0; p < PC; ++p) q[c][p] = img[(c - C0) * W + x0 + p];
    }
    template <int W, int C0>
    __device__ __forceinline__ void halo_half(const T* img)
    {
        static_assert(xs<W>() >= 2 && xs<W>() + 64 * PC + 2 <= W, "halo inside the node");
#pragma unroll
        for (int c = C0; c < C0 + 3; ++c) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                hl[c][i] = img[(c - C0) * W + xs<W>() - 1 - i];
                hr[c][i] = img[(c - C0) * W + xs<W>() + 64 * PC + i];
            }
        }
    }
    // the region's cells to the state arrays
    template <int W>
    __device__ __forceinline__ void store_global(T* out, int64_t n, int64_t base, int lane) const
    {
        const int x0 = xs<W>() + lane * PC;
#pragma unroll
        for (int c = 0; c < 6; ++c)
#pragma unroll
            for (int p = 0; p < PC; ++p) out[c * n + wrap(base + x0 + p, n)] = q[c][p];
    }
};

// Ring PC's cells of components C0 .. C0+2: from the state arrays into a
// three-component node image, and from the image to the state arrays.
template <typename T, int W, int PC, int C0>
__device__ __forceinline__ void eu_ring_in(T* img, const T* in, int64_t n, int64_t base, int lane)
{
    const int x = ring_x<W, PC>(lane);
#pragma unroll
    for (int c = C0; c < C0 + 3; ++c) img[(c - C0) * W + x] = in[c * n + wrap(base + x, n)];
}
template <typename T, int W, int PC, int C0>
__device__ __forceinline__ void eu_ring_out(const T* img, T* out, int64_t n, int64_t base, int lane)
{
    const int x = ring_x<W, PC>(lane);
#pragma unroll
    for (int c = C0; c < C0 + 3; ++c) out[c * n + wrap(base + x, n)] = img[(c - C0) * W + x];
}

// Smallest region of the phased Euler tiles, in cells per lane.
constexpr int kEuRegionFirst = 1;

// A phased Euler tile's node: its base in the state arrays and the wave's
// three-component LDS image (3 W values).
template <typename T>
struct EuNode {
    T* img;
    const T* in;
    T* out;
    int64_t n, base;
    int lane;
};

// Region A -> region B = A + 1 cells per lane (B = W/64: the whole node), one
// half of the state at a time through the image.  The cells of ring B, and
// the halo of region B, lie outside every region so far, so they still hold
// the tile's input.
template <typename T, int W, int A, int B>
__device__ __forceinline__ void eu_grow(const EulerRegion<T, A>& a, EulerRegion<T, B>& b, const EuNode<T>& d)
{
    for_each_index(
        [&](auto h) {
            constexpr int C0 = 3 * decltype(h)::value;
            a.template save_half<W, C0>(d.img, d.lane);
            eu_ring_in<T, W, B, C0>(d.img, d.in, d.n, d.base, d.lane);
            wave_sync();
            b.template load_half<W, C0>(d.img, d.lane);
            wave_sync();
        },
        std::make_integer_sequence<int, 2>{});
    b.template halo_global<W>(d.in, d.n, d.base);
    b.place(W, EulerRegion<T, B>::template xs<W>() + d.lane * B, d.base, d.n);
}

// Region A -> region B = A - 1 cells per lane: ring A is final and goes to
// the output; region B's halo lies in ring A and comes from the image.
template <typename T, int W, int A, int B>
__device__ __forceinline__ void eu_shrink(const EulerRegion<T, A>& a, EulerRegion<T, B>& b, const EuNode<T>& d)
{
    for_each_index(
        [&](auto h) {
            constexpr int C0 = 3 * decltype(h)::value;
            a.template save_half<W, C0>(d.img, d.lane);
            wave_sync();
            eu_ring_out<T, W, A, C0>(d.img, d.out, d.n, d.base, d.lane);
            b.template load_half<W, C0>(d.img, d.lane);
            b.template halo_half<W, C0>(d.img);
            wave_sync();
        },
        std::make_integer_sequence<int, 2>{});
    b.place(W, EulerRegion<T, B>::template xs<W>() + d.lane * B, d.base, d.n);
}

// The down phase from region PC (loaded) on: region PC takes down pairs
// 16 PC - 15 <= s <= 16 PC - 1 (from 1 for the first region), where every
// threshold is <= 64 PC - 1; the whole node ends it in `full`.
template <typename T, int P, int PC>
__device__ __forceinline__ void eu_down(EulerRegion<T, PC>& r, EulerRegion<T, P>& full, const EuNode<T>& d,
                                        const EulerCoef<T>& k)
{
    constexpr int W = kWave * P, H = W / 4;
    r.down(PC == kEuRegionFirst ? 1 : 16 * PC - 15, 16 * PC - 1, k);
    if constexpr (PC + 1 < P) {
        EulerRegion<T, PC + 1> r2;
        eu_grow<T, W, PC, PC + 1>(r, r2, d);
        eu_down<T, P, PC + 1>(r2, full, d, k);
    } else {
        eu_grow<T, W, PC, P>(r, full, d);
        full.down(16 * (P - 1) + 1, H - 1, k);
    }
}

// The up phase from region PC + 1 (or the whole node, PC + 1 = P) down:
// region PC takes up pairs 16(P-PC)+1 <= m <= 16(P-PC)+15 (to H-3 for the
// first region); each ring goes to the output once final, the first region
// last.
template <typename T, int P, int PC>
__device__ __forceinline__ void eu_up(const EulerRegion<T, PC + 1>& a, const EuNode<T>& d, const EulerCoef<T>& k)
{
    constexpr int W = kWave * P, H = W / 4;
    EulerRegion<T, PC> b;
    eu_shrink<T, W, PC + 1, PC>(a, b, d);
    if constexpr (PC == kEuRegionFirst) {
        b.up(W, 16 * (P - PC) + 1, H - 3, k);
        b.template stage<0, false>(W - 1 - 4 * (H - 1), k);
        b.template store_global<W>(d.out, d.n, d.base, d.lane);
    } else {
        b.up(W, 16 * (P - PC) + 1, 16 * (P - PC) + 15, k);
        eu_up<T, P, PC - 1>(b, d, k);
    }
}

// Swept Euler tiles: one wave per node of W = 64*P cells.  For P >= 4 the
// diamond's levels run on the narrowest centred region of 1, 2, .. P cells
// per lane that holds their active set and the two-cell stencil reach (same
// operations, same bits), and a change of region moves the lane's cells
// through an LDS image of three of the six components at a time: 12 KB per
// wave at W = 512, so that two waves fit on a SIMD (the kernel is held to
// 256 registers for the same reason).  The node's cells come from the input
// ring by ring as the regions grow and go to the output ring by ring as they
// shrink.
template <typename T, int P, int TILE>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2)))
void k_euler_swept(const T* __restrict__ in, T* __restrict__ out, int64_t n, int64_t nnodes,
                   int64_t node_first, int64_t offset, EulerCoef<T> k)
{
    constexpr int W = kWave * P, H = W / 4;
    constexpr bool PHASED = P >= 4;
    __shared__ T img_all[PHASED ? kWavesPerBlock * 3 * W : 1];
    NodeGeom g;
    if (!node_geom<P>(n, nnodes, node_first, offset, g)) return;

    EulerRegion<T, P> full;
    if constexpr (!PHASED) {
        full.template load_global<W>(in, n, g.base, g.lane);
        full.place(W, g.lane * P, g.base, n);
        if (TILE != TILE_UP) full.down(1, H - 1, k);
        if (TILE != TILE_DOWN) {
            full.up(W, 1, H - 3, k);
            full.template stage<0, false>(W - 1 - 4 * (H - 1), k);
        }
        full.template store_global<W>(out, n, g.base, g.lane);
    } else {
        constexpr int F = kEuRegionFirst;
        const EuNode<T> d{img_all + (threadIdx.x >> 6) * 3 * W, in, out, n, g.base, g.lane};
        if (TILE != TILE_UP) {
            EulerRegion<T, F> r;
            r.template load_global<W>(in, n, g.base, g.lane);
            r.place(W, EulerRegion<T, F>::template xs<W>() + g.lane * F, g.base, n);
            eu_down<T, P, F>(r, full, d, k);
        } else {
            full.template load_global<W>(in, n, g.base, g.lane);
            full.place(W, g.lane * P, g.base, n);
        }
        if (TILE != TILE_DOWN) {
            full.up(W, 1, 15, k);
            eu_up<T, P, P - 1>(full, d, k);
        } else {
            full.template store_global<W>(out, n, g.base, g.lane);
        }
    }
}

// ------------------------------------------------------ classic kernels ---
// Euler classic stage (Euler:391-426) with each interface flux evaluated once:
// lane l of a wave computes the interface between cells x = 63 w + l - 1 and
// x + 1, and (l < 63) updates cell x + 1 from it and from lane l + 1's,
// which a DPP shift brings: 63 cells per wave, and the values the per-cell
// form computes twice, so the same bits.  Cell indices are clamped at the
// domain ends as in the per-cell form (the values so read are unused there).
template <typename T, int STAGE>
__global__ __launch_bounds__(kClassicBlock) void k_euler_classic(T* __restrict__ buf, int64_t n,
                                                                 EulerCoef<T> k)
{
    constexpr int src = STAGE == 0 ? 0 : 3, dst = 3 - src;
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t wave = (int64_t)blockIdx.x * (kClassicBlock / kWave) + (threadIdx.x >> 6);
    const int64_t x = wave * (kWave - 1) + lane - 1;
    auto cell = [&](int64_t j) {
        j = j < 0 ? 0 : (j > n - 1 ? n - 1 : j);
        return Q3<T>{buf[(src + 0) * n + j], buf[(src + 1) * n + j], buf[(src + 2) * n + j]};
    };
    const Q3<T> A = cell(x - 1), B = cell(x), C = cell(x + 1), Dc = cell(x + 2);
    // the interface right of cell 0 drops pdiff(-1,0), the one left of cell
    // n-1 drops pdiff(n-1,n) (the flags of Euler:405, :424)
    const T q0 = x == 0 ? T(0) : eu_pdiff(A, B);
    const T q1 = eu_pdiff(B, C);
    const T q2 = x == n - 2 ? T(0) : eu_pdiff(C, Dc);
    Q3<T> FL, DL;
    eu_iface<Ieee<T>>(A, B, C, Dc, q0, q1, q2, k, FL, DL);
    // every lane takes part in the shifts before any leaves
    const Q3<T> FR{from_right(FL.x, FL.x), from_right(FL.y, FL.y), from_right(FL.z, FL.z)};
    const Q3<T> DR{from_right(DL.x, DL.x), from_right(DL.y, DL.y), from_right(DL.z, DL.z)};
    const int64_t i = x + 1;
    if (lane == kWave - 1 || i >= n) return;
    Q3<T> nv;
    if (i == 0) {
        nv = k.bl;
    } else if (i == n - 1) {
        nv = k.br;
    } else {
        const Q3<T> f = eu_balance(FL, DL, FR, DR);
        if (STAGE == 0)
            nv = eu_apply(C, f, T(0.25) * k.dtdx);
        else
            nv = eu_apply(Q3<T>{buf[i], buf[n + i], buf[2 * n + i]}, f, T(0.5) * k.dtdx);
    }
    buf[(dst + 0) * n + i] = nv.x;
    buf[(dst + 1) * n + i] = nv.y;
    buf[(dst + 2) * n + i] = nv.z;
}

// ------------------------------------------------------------- dispatch ---
template <typename T> const EulerCoef<T>& eu_of(const Coefs& c);
template <> const EulerCoef<double>& eu_of<double>(const Coefs& c) { return c.eu_d; }
template <> const EulerCoef<float>& eu_of<float>(const Coefs& c) { return c.eu_f; }

template <typename T, int P, int TILE>
hipError_t swept_tile(const SweptLaunch& L, const Coefs& c, hipStream_t s)
{
    const int64_t count = L.nnodes - L.node_first;
    if (count <= 0) return hipSuccess;
    const dim3 grid((unsigned)((count + kWavesPerBlock - 1) / kWavesPerBlock));
    hipLaunchKernelGGL((k_euler_swept<T, P, TILE>), grid, dim3(kBlock), 0, s, static_cast<const T*>(L.in),
                       static_cast<T*>(L.out), L.n, L.nnodes, L.node_first, L.offset, eu_of<T>(c));
    return hipGetLastError();
}

template <typename T, int P>
hipError_t swept_points(const SweptLaunch& L, const Coefs& c, hipStream_t s)
{
    switch (L.tile) {
    case TILE_UP: return swept_tile<T, P, TILE_UP>(L, c, s);
    case TILE_DOWN: return swept_tile<T, P, TILE_DOWN>(L, c, s);
    case TILE_DIAMOND: return swept_tile<T, P, TILE_DIAMOND>(L, c, s);
    }
    return hipErrorInvalidValue;
}

template <typename T>
hipError_t swept_prec(const SweptLaunch& L, const Coefs& c, hipStream_t s)
{
    switch (L.P) {
    case 1: return swept_points<T, 1>(L, c, s);
    case 2: return swept_points<T, 2>(L, c, s);
    case 4: return swept_points<T, 4>(L, c, s);
    case 8: return swept_points<T, 8>(L, c, s);
    }
    return hipErrorInvalidValue;
}

template <typename T>
hipError_t stage_prec(int stage, int64_t n, void* buf, const Coefs& c, hipStream_t s)
{
    T* b = static_cast<T*>(buf);
    const int64_t waves = (n + kWave - 2) / (kWave - 1);  // 63 cells per wave
    const dim3 grid((unsigned)((waves + kClassicBlock / kWave - 1) / (kClassicBlock / kWave)));
    if (stage == 0)
        hipLaunchKernelGGL((k_euler_classic<T, 0>), grid, dim3(kClassicBlock), 0, s, b, n, eu_of<T>(c));
    else
        hipLaunchKernelGGL((k_euler_classic<T, 1>), grid, dim3(kClassicBlock), 0, s, b, n, eu_of<T>(c));
    return hipGetLastError();
}

}  // namespace

hipError_t launch_swept_euler(const SweptLaunch& L, bool f64, const Coefs& c, hipStream_t s)
{
    return f64 ? swept_prec<double>(L, c, s) : swept_prec<float>(L, c, s);
}

hipError_t launch_stage_euler(bool f64, int stage, int64_t n, void* buf, const Coefs& c, hipStream_t s)
{
    return f64 ? stage_prec<double>(stage, n, buf, c, s) : stage_prec<float>(stage, n, buf, c, s);
}

}  // namespace sw1d
