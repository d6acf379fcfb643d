// Batched solve: many independent periodic heat / KS problems of arbitrary
// sizes advanced together, as workgroup-wide overlapped tiles (sw1d_wide.hpp).
//
// A launch advances every problem of a group (one equation, one tile shape) by
// the same number of steps; its workgroups are the group's tiles, found in a
// table made on the host, so a large problem spreads over as many compute
// units as its size asks for.  A table serves any number of steps: a launch may
// take as many as the group's widest tile leaves its window (BatchGroup::cap).
// (A workgroup per problem, stepping it through
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
    Coef<T, EQ> k;
    if constexpr (EQ == EQ_HEAT)
        k = {J.c[0], J.c[1]};
    else
        k = {KsCoef<T>{J.c[0], J.c[1], J.c[2], J.c[3], J.c[4]}};
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

// One of every `stride` of the problems named, for estimates: an advance by a new
// number of steps makes some hundred of them.  Which one varies from stride to
// stride (a generator of its own, so the same every time): sizes in a pattern that
// repeats would otherwise be sampled at one place of it.
BatchSample sample_of(const std::vector<int64_t>& n, const std::vector<int>& at)
{
    BatchSample s;
    const size_t stride = (at.size() + 255) / 256;
    uint32_t pick = 1;
    for (size_t j = 0; j < at.size(); j += stride) {
        pick = pick * 1664525u + 1013904223u;  // Numerical Recipes' linear congruential generator
        s.n.push_back(n[at[j + (pick >> 16) % std::min(stride, at.size() - j)]]);
    }
    if (!s.n.empty()) s.weight = (double)at.size() / (double)s.n.size();
    return s;
}

// Tiles of at most `most` points that the problems need.
double tiles_of(const BatchSample& g, double most)
{
    double t = 0;
    for (int64_t n : g.n) t += std::ceil((double)n / most);
    return t * g.weight;
}

// The cost model of wide_choose for launches of `tiles` tiles and `each` steps.
double group_us(const Cost& c, double tiles, double launches, double each, int cus)
{
    const double m = std::ceil(tiles / cus);
    return launches * (c.t0 + (m - 1) * c.t2 + each * (c.c1 + (m - 1) * c.c2));
}
double even_launches(double nsteps, double most) { return 2 * std::ceil(nsteps / (2 * most)); }

// The steps per launch that take a group the least time, and that time.
struct Timing { double us = 0; int steps = 0; };
Timing time_group(int eq, bool f64, int shape, const BatchSample& g, int64_t nsteps, int cus)
{
    const Entry& e = entries(eq)[shape];
    const Cost& c = f64 ? e.f64 : e.f32;
    const int win = window(e), r = reach(eq);
    Timing best;
    for (double f : {.95, .9, .85, .8, .75, .7, .6, .45, .3}) {
        const double s = std::floor((1 - f) * win / (2 * r));
        if (s < 1) continue;
        const double launches = even_launches((double)nsteps, s), each = std::ceil(nsteps / launches);
        const double us = group_us(c, tiles_of(g, win - 2 * r * each), launches, each, cus);
        if (best.steps == 0 || us < best.us) best = Timing{us, (int)each};
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
    // by points per tile; those that store fewer points in more time never win
    std::stable_sort(v.begin(), v.end(), [](const ShapeCost& a, const ShapeCost& b) {
        return a.per_tile != b.per_tile ? a.per_tile < b.per_tile : a.us < b.us;
    });
    std::vector<ShapeCost> kept;
    for (const ShapeCost& k : v)
        if (kept.empty() || k.us < kept.back().us) kept.push_back(k);
    return kept;
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

std::vector<int> problems_of(const std::vector<int32_t>& eq, int e)
{
    std::vector<int> all;
    for (size_t i = 0; i < eq.size(); ++i)
        if (eq[i] == e) all.push_back((int)i);
    return all;
}

// One shape for every problem of an equation (few problems: the chip is not
// full), or each problem's own, whichever takes less time by the sample.
struct Choice { double us = 0; int shape = -1; };  // shape < 0: each its own
Choice choose(int e, bool f64, const BatchSample& s, const std::vector<ShapeCost>& costs, int64_t nsteps, int cus)
{
    Choice best;
    for (int i = 0; i < shapes(e); ++i) {
        const Timing t = time_group(e, f64, i, s, nsteps, cus);
        if (t.steps && (best.shape < 0 || t.us < best.us)) best = Choice{t.us, i};
    }
    std::vector<BatchSample> own((size_t)shapes(e));
    for (int64_t n : s.n) own[(size_t)shape_for(costs, n)].n.push_back(n);
    double sum = 0;
    for (int i = 0; i < shapes(e); ++i) {
        own[i].weight = s.weight;
        if (!own[i].n.empty()) sum += time_group(e, f64, i, own[i], nsteps, cus).us;
    }
    return sum < best.us ? Choice{sum, -1} : best;
}

}  // namespace

hipError_t launch_batch(const BatchLaunch& L, bool f64, hipStream_t s)
{
    return f64 ? launch_prec<double>(L, s) : launch_prec<float>(L, s);
}

int64_t BatchGroup::launches(int64_t nsteps) const { return 2 * ((nsteps + 2 * cap - 1) / (2 * cap)); }

double batch_us(const std::vector<BatchGroup>& groups, bool f64, int64_t nsteps, int cus)
{
    double us = 0;
    for (const BatchGroup& g : groups) {
        const Entry& e = entries(g.eq)[g.shape];
        const double launches = (double)g.launches(nsteps), each = std::ceil(nsteps / launches);
        us += group_us(f64 ? e.f64 : e.f32, (double)g.ntiles, launches, each, cus);
    }
    return us;
}

BatchSample batch_sample(const std::vector<int32_t>& eq, const std::vector<int64_t>& n, int e)
{
    return sample_of(n, problems_of(eq, e));
}

double batch_least_us(const BatchSample (&s)[2], bool f64, int64_t nsteps, int cus)
{
    double us = 0;
    for (int e = EQ_HEAT; e <= EQ_KS; ++e)
        if (!s[e].n.empty()) us += choose(e, f64, s[e], shape_costs(e, f64, nsteps), nsteps, cus).us;
    return us;
}

void batch_groups(const std::vector<int32_t>& eq, const std::vector<int64_t>& n, bool f64, int64_t nsteps, int cus,
                  std::vector<BatchGroup>& groups, std::vector<BatchTile>& tiles)
{
    groups.clear();
    tiles.clear();
    for (int e = EQ_HEAT; e <= EQ_KS; ++e) {
        std::vector<int> all = problems_of(eq, e);
        if (all.empty()) continue;
        const std::vector<ShapeCost> costs = shape_costs(e, f64, nsteps);
        const Choice c = choose(e, f64, sample_of(n, all), costs, nsteps, cus);
        std::vector<std::vector<int>> own((size_t)shapes(e));
        if (c.shape < 0) {
            std::vector<int8_t> known(1 << 16, -1);  // shapes of the sizes below, as they are met
            for (int i : all) {
                int8_t* k = n[i] < (int64_t)known.size() ? &known[(size_t)n[i]] : nullptr;
                const int shape = k && *k >= 0 ? *k : shape_for(costs, n[i]);
                if (k) *k = (int8_t)shape;
                own[(size_t)shape].push_back(i);
            }
        } else {
            own[(size_t)c.shape] = std::move(all);
        }
        for (int i = 0; i < shapes(e); ++i) {
            if (own[i].empty()) continue;
            BatchGroup g;
            g.eq = e;
            g.shape = i;
            g.first = (int64_t)tiles.size();
            const int64_t win = window(entries(e)[i]), r = reach(e);
            const int64_t most = win - 2 * r * time_group(e, f64, i, sample_of(n, own[i]), nsteps, cus).steps;
            int64_t widest = 1;
            for (int j : own[i]) {
                const int64_t k = (n[j] + most - 1) / most, w = (n[j] + k - 1) / k;
                widest = std::max(widest, w);
                for (int64_t o = 0; o < n[j]; o += w)
                    tiles.push_back(BatchTile{j, (int32_t)o, (int32_t)std::min(w, n[j] - o)});
            }
            g.ntiles = (int64_t)tiles.size() - g.first;
            g.cap = (win - widest) / (2 * r);
            groups.push_back(g);
        }
    }
}

}  // namespace sw1d
