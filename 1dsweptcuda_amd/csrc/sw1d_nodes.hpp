// Node geometry and small helpers shared by the swept tile kernels
// (sw1d_kernels.hip, sw1d_euler.hip).
#pragma once

#include <type_traits>
#include <utility>

#include "sw1d_internal.hpp"
#include "sw1d_lanes.hpp"

namespace sw1d {
namespace {

constexpr int kWavesPerBlock = 4;
constexpr int kBlock = kWave * kWavesPerBlock;
constexpr int kClassicBlock = 256;


template <typename T, int P>
__device__ __forceinline__ void load_pts(const T* __restrict__ a, int64_t i0, T (&v)[P])
{
#pragma unroll
    for (int p = 0; p < P; ++p) v[p] = a[i0 + p];
}
template <typename T, int P>
__device__ __forceinline__ void store_pts(T* __restrict__ a, int64_t i0, const T (&v)[P])
{
#pragma unroll
    for (int p = 0; p < P; ++p) a[i0 + p] = v[p];
}

struct NodeGeom {
    int64_t base;  // global index of node-local x = 0
    int64_t lb;    // global index of this lane's first point
    int lane;
};

template <int P>
__device__ __forceinline__ bool node_geom(int64_t n, int64_t nnodes, int64_t node_first,
                                          int64_t offset, NodeGeom& g)
{
    constexpr int W = kWave * P;
    g.lane = threadIdx.x & (kWave - 1);
    const int64_t node = node_first + (int64_t)blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
    if (node >= nnodes) return false;
    int64_t b = node * W + offset;
    b = b >= n ? b - n : b;
    g.base = b;
    int64_t lb = b + (int64_t)g.lane * P;
    g.lb = lb >= n ? lb - n : lb;
    return true;
}

__device__ __forceinline__ int64_t wrap(int64_t i, int64_t n)
{
    return i < 0 ? i + n : (i >= n ? i - n : i);
}

// Calls f(integral_constant<int, i>) for i = 0, 1, .. in order.
template <typename F, int... I>
__device__ __forceinline__ void for_each_index(F&& f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}

// Calls f(integral_constant<int, j>) for j = A, A + 1, .. B in order (none if A > B).
template <int A, int B, typename F>
__device__ __forceinline__ void for_range(F&& f)
{
    if constexpr (A <= B) {
        f(std::integral_constant<int, A>{});
        for_range<A + 1, B>(f);
    }
}

// Ring PC of a node (1 <= PC <= P) is the 64 points that the centred region
// of PC points per lane holds and the region of PC - 1 does not: 32 on each
// side of the centre.  Lane l takes ring point l, so a ring moves between HBM
// and the LDS image as two coalesced 256-byte runs per state array.
template <int W, int PC>
__device__ __forceinline__ int ring_x(int lane)
{
    return lane < 32 ? W / 2 - 32 * PC + lane : W / 2 + 32 * (PC - 1) + (lane - 32);
}

// Orders a wave's own LDS writes before its own reads of other lanes' data:
// LDS executes a wave's instructions in order, and the wavefront-scope
// fences keep the compiler from moving one lane's loads above other lanes'
// stores.  Each wave of the tile kernels owns its slice of the LDS image.
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace
}  // namespace sw1d
