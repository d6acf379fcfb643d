// Batched solve: many independent periodic heat / KS problems of arbitrary
// sizes advanced together, as workgroup-wide overlapped tiles (sw1d_wide.hpp).
//
// A launch advances every problem of a group (one equation, one tile shape) by
// the same number of steps; its workgroups are the group's tiles, found in a
// table made on the host, so a large problem spreads over as many compute
// units as its size asks for.  (A workgroup per problem, stepping it through
// the whole advance, was bound by the largest one: 512 problems of 2^10 .. 2^16
// points, 5000 steps, FP64, took 70 ms, 51 ms of them one workgroup's.)  Every
// group's launches come in an even number, so its result is back in the
// buffer it started from.

#include <algorithm>
#include <cmath>

#include "sw1d_wide.hpp"

namespace sw1d {
namespace {

using namespace wide;

template <typename T, int EQ, class S>
__global__ __launch_bounds__(S::NT) void k_batch(const BatchTile* __restrict__ tiles,
                                                 const BatchJob<T>* __restrict__ jobs, const T* __restrict__ in,
                                                 T* __restrict__ out, int steps)
{
    __shared__ __attribute__((aligned(16))) T lds[S::template lds<T>];
    const BatchTile t = tiles[blockIdx.x];
    const BatchJob<T>& J = jobs[t.job];
    Coef<T> k;
    k.fo = J.c[0];
    k.fo2 = J.c[1];
    k.ks = KsCoef<T>{J.c[0], J.c[1], J.c[2], J.c[3], J.c[4]};
    tile<T, EQ, S>(lds, in + J.offset, out + J.offset, J.n, 0, t.out0, t.count, steps, ENDS_PERIODIC, k);
}

template <typename T, int EQ, int I = 0>
hipError_t launch_group(const BatchLaunch& L, hipStream_t s)
{
    if constexpr (I < Table<EQ>::count) {
        if (L.shape != I) return launch_group<T, EQ, I + 1>(L, s);
        using S = TableShape<EQ, I>;
        hipLaunchKernelGGL((k_batch<T, EQ, S>), dim3((unsigned)L.ntiles), dim3(S::NT), 0, s, L.tiles,
                           static_cast<const BatchJob<T>*>(L.jobs), static_cast<const T*>(L.in),
                           static_cast<T*>(L.out), L.steps);
        return hipGetLastError();
    } else {
        return hipErrorInvalidValue;
    }
}

template <typename T>
hipError_t launch_prec(const BatchLaunch& L, hipStream_t s)
{
    return L.eq == EQ_HEAT ? launch_group<T, EQ_HEAT>(L, s) : launch_group<T, EQ_KS>(L, s);
}

// A group's launches and steps per launch (the longer ones), and their time.
struct Timing { double us = 0; int64_t launches = 0; int steps = 0; };

// Tiles of at most `most` points that the members need (from a sample of large
// groups: the estimate is made some hundred times per new step count).
double tiles_of(const std::vector<int64_t>& n, const std::vector<int>& members, double most)
{
    const size_t stride = (members.size() + 255) / 256;
    double t = 0;
    size_t seen = 0;
    for (size_t j = 0; j < members.size(); j += stride, ++seen) t += std::ceil((double)n[members[j]] / most);
    return t * (double)members.size() / (double)seen;
}

// The best steps per launch of a group: the cost model of wide_choose with the
// group's tiles and an even number of launches.
Timing time_group(int eq, bool f64, int shape, const std::vector<int64_t>& n, const std::vector<int>& members,
                  int64_t nsteps, int cus)
{
    const Entry& e = entries(eq)[shape];
    const Cost& c = f64 ? e.f64 : e.f32;
    const int win = window(e), r = reach(eq);
    Timing best;
    for (double f : {.95, .9, .85, .8, .75, .7, .6, .45, .3}) {
        const double s = std::floor((1 - f) * win / (2 * r));
        if (s < 1) continue;
        const double launches = 2 * std::ceil((double)nsteps / (2 * s)), each = std::ceil(nsteps / launches);
        const double m = std::ceil(tiles_of(n, members, win - 2 * r * each) / cus);
        const double us = launches * (c.t0 + (m - 1) * c.t2 + each * (c.c1 + (m - 1) * c.c2));
        if (best.launches == 0 || us < best.us) best = Timing{us, (int64_t)launches, (int)each};
    }
    return best;
}

// A problem's own best shape where every compute unit is busy anyway: the
// least time per step of its tiles' throughput.
struct ShapeCost { int shape; double per_tile, us; };  // 1 / (points a tile stores), us per step and tile
std::vector<ShapeCost> shape_costs(int eq, bool f64, int64_t nsteps)
{
    std::vector<ShapeCost> v;
    for (int i = 0; i < shapes(eq); ++i) {
        const Entry& e = entries(eq)[i];
        const Cost& c = f64 ? e.f64 : e.f32;
        const int win = window(e), r = reach(eq);
        for (double f : {.95, .9, .85, .8, .7, .6, .45, .3}) {
            const double s = std::min(std::floor((1 - f) * win / (2 * r)), (double)nsteps);
            // the launch itself, spread over four tiles per compute unit
            if (s >= 1) v.push_back({i, 1.0 / (win - 2 * r * s), c.c2 + (c.t2 + c.t0 / 4) / s});
        }
    }
    return v;
}
int shape_for(const std::vector<ShapeCost>& costs, int64_t n)
{
    int best = 0;
    double least = 0;
    for (const ShapeCost& k : costs) {
        const double us = std::ceil((double)n * k.per_tile) * k.us;
        if (least == 0 || us < least) {
            least = us;
            best = k.shape;
        }
    }
    return best;
}

}  // namespace

hipError_t launch_batch(const BatchLaunch& L, bool f64, hipStream_t s)
{
    return f64 ? launch_prec<double>(L, s) : launch_prec<float>(L, s);
}

void batch_groups(const std::vector<int32_t>& eq, const std::vector<int64_t>& n, bool f64, int64_t nsteps, int cus,
                  std::vector<BatchGroup>& groups, std::vector<BatchTile>& tiles)
{
    groups.clear();
    tiles.clear();
    if (cus <= 0) cus = 256;
    for (int e = EQ_HEAT; e <= EQ_KS; ++e) {
        std::vector<int> all;
        for (size_t i = 0; i < n.size(); ++i)
            if (eq[i] == e) all.push_back((int)i);
        if (all.empty()) continue;
        // one shape for every problem (few problems: the chip is not full) ...
        int shape = 0;
        Timing best;
        for (int i = 0; i < shapes(e); ++i) {
            const Timing t = time_group(e, f64, i, n, all, nsteps, cus);
            if (t.launches && (best.launches == 0 || t.us < best.us)) {
                best = t;
                shape = i;
            }
        }
        // ... or each problem's own
        std::vector<std::vector<int>> own((size_t)shapes(e));
        const std::vector<ShapeCost> costs = shape_costs(e, f64, nsteps);
        for (int i : all) own[(size_t)shape_for(costs, n[i])].push_back(i);
        std::vector<Timing> each((size_t)shapes(e));
        double sum = 0;
        for (int i = 0; i < shapes(e); ++i)
            if (!own[i].empty()) {
                each[i] = time_group(e, f64, i, n, own[i], nsteps, cus);
                sum += each[i].us;
            }
        if (sum >= best.us) {
            for (auto& m : own) m.clear();
            own[shape] = all;
            each[shape] = best;
        }
        for (int i = 0; i < shapes(e); ++i) {
            if (own[i].empty()) continue;
            BatchGroup g;
            g.eq = e;
            g.shape = i;
            g.launches = each[i].launches;
            g.first = (int64_t)tiles.size();
            const int64_t most = window(entries(e)[i]) - 2 * (int64_t)reach(e) * each[i].steps;
            for (int j : own[i]) {
                const int64_t k = (n[j] + most - 1) / most, w = (n[j] + k - 1) / k;
                for (int64_t o = 0; o < n[j]; o += w)
                    tiles.push_back(BatchTile{j, (int32_t)o, (int32_t)std::min(w, n[j] - o)});
            }
            g.ntiles = (int64_t)tiles.size() - g.first;
            groups.push_back(g);
        }
    }
}

}  // namespace sw1d
