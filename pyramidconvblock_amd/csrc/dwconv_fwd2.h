// The forward convolutions of both scales of a two-scale block as one launch: y0 = conv(x0, w0) at the full scale and
// y1 = conv(x1, w1) at the pooled one (x1 being the average pool of x0, made before the launch), neither
// depending on the other.  A compute unit holds one workgroup of these kernels at a time and a run of rows costs a start-up
// that does not depend on its length, so a launch of its own cuts a problem into enough runs to fill the chip; here each
// scale gets the part of the chip that lets both end together.  us a launch, 20 of them in a graph: [32,56,56,64] filter 13 15.1
// (bands of one image instead of runs 15.4), 17 20.1 (22.8), [128,56,56,64] filter 13 39 (41), 17 55.5 (68); the two launches
// one by one at [32,56,56,64] filter 13 12.2 + 8.0 and a gap.  Each scale runs in the tile
// (16 or 8 patches side by side) that its width fills better: by template where the full scale's is the wide one and slices
// are 16 channels (each workgroup starts with one problem's arguments and no choice between the fields of two; at run time,
// us: filter 13 15.4 for 15.0, 9 14.2 for 13.95), at run time elsewhere (filters 15 and 17, whose slices are 8 channels: by
// template no faster when measured with bands).
// The kernel template and its per-filter-size launcher; dwconv_fwd2_k<K>.hip instantiate it, one file per size.
#pragma once
#include <algorithm>
#include <functional>
#include <map>
#include <tuple>
#include <type_traits>
#include <vector>

#include "dwconv_tz.h"
#include "pool_branch.h"

namespace pdw {

struct Fwd2Problem {
    const void *x, *w;
    void* y;
    TzGeom g;
    int npc;       // patches of a tile side by side
    int start, n;  // first workgroup and number of workgroups
};

struct Fwd2Args {
    Fwd2Problem p[2];
    PoolFwdJob mean;      // workgroups behind both problems (one per image, mean.B of them): the block's mean branch
};

// MODE 0: the convolutions; 4: each with the gate applied in its store (dwconv_tz.h).
// NPC0, NPC1: patches side by side of the two problems' tiles; 0: as the arguments say.
template <typename T, int K, int CS, int NPC0, int NPC1, int MODE>
__global__ __launch_bounds__(512, 1) void dwconv_fwd2_k(const Fwd2Args a) {
    const int blk = blockIdx.x;
    if constexpr (NPC0 != 0) {
        if ((unsigned)(blk - a.p[0].start) < (unsigned)a.p[0].n) {
            dwconv_tz_body<T, K, NPC0, CS, MODE>((const T*)a.p[0].x, (const T*)a.p[0].w, nullptr, nullptr, (T*)a.p[0].y, a.p[0].g,
                                                 blk - a.p[0].start, a.p[0].n);
            return;
        }
        if ((unsigned)(blk - a.p[1].start) < (unsigned)a.p[1].n) {
            dwconv_tz_body<T, K, NPC1, CS, MODE>((const T*)a.p[1].x, (const T*)a.p[1].w, nullptr, nullptr, (T*)a.p[1].y, a.p[1].g,
                                                 blk - a.p[1].start, a.p[1].n);
            return;
        }
    }
    if (NPC0 != 0 || blk >= a.p[0].n + a.p[1].n) {
        // The mean branch (per-image mean -> conv_pool -> the row added to every output row of the image) needs a
        // launch whose memory system is not saturated, and its inputs are ready when this one starts: last in the
        // grid, its short workgroups go to compute units the convolutions leave free or have finished with.
        extern __shared__ uint32_t smem[];
        pool_branch_fwd_v8_body<T>(a.mean.part, a.mean.nchunks, a.mean.D, a.mean.inv_p, (const T*)a.mean.wp,
                                   (const T*)a.mean.bp, (const T*)a.mean.bo, (T*)a.mean.m, a.mean.rowbias,
                                   blk - a.p[0].n - a.p[1].n, reinterpret_cast<float*>(smem));
        return;
    }
    if constexpr (NPC0 == 0) {
        const bool first = (unsigned)(blk - a.p[0].start) < (unsigned)a.p[0].n;
        const T* const x = (const T*)(first ? a.p[0].x : a.p[1].x);
        const T* const w = (const T*)(first ? a.p[0].w : a.p[1].w);
        T* const y = (T*)(first ? a.p[0].y : a.p[1].y);
        const TzGeom g = first ? a.p[0].g : a.p[1].g;
        const int at = blk - (first ? a.p[0].start : a.p[1].start), n = first ? a.p[0].n : a.p[1].n;
        if ((first ? a.p[0].npc : a.p[1].npc) == 16)
            dwconv_tz_body<T, K, 16, CS, MODE>(x, w, nullptr, nullptr, y, g, at, n);
        else
            dwconv_tz_body<T, K, 8, CS, MODE>(x, w, nullptr, nullptr, y, g, at, n);
    }
}

// One way of cutting a problem of a shared launch: pieces (runs of rows, bands per image), time and number of its workgroups.
struct LaunchCut {
    int n;
    double cost;
    long long count;
};

// The time the last workgroup ends when the problems' workgroups, in the order `ord`, go to the earliest free of 256 compute
// units (these kernels' workgroups have one to themselves).
template <int N>
inline double launch_makespan(const LaunchCut* const (&cuts)[N], const int (&ord)[N]) {
    std::map<double, long long> free_at{{0.0, 256}};   // compute units by the time they are free at
    double end = 0;
    long long total = 0;
    for (int o : ord) {
        const LaunchCut& c = *cuts[o];
        total += c.count;
        for (long long left = c.count; left > 0;) {
            const auto first = free_at.begin();
            const double t = first->first + c.cost;
            const long long n = std::min(left, first->second);
            left -= n, end = std::max(end, t);
            if ((first->second -= n) == 0) free_at.erase(first);
            free_at[t] += n;
        }
    }
    return total > 256 ? 1.05 * end : end;   // (several rounds end later than that: see launch_balance)
}

// A problem that can be cut into runs of at most a number of steps: time of a run = start + step x its steps.
struct LaunchPart {
    double start, step;
    int total, least;                        // steps of the whole problem; fewest of a run
    std::function<long long(int)> blocks;    // workgroups when cut so
};
constexpr double kMeanCost = 8.0;   // us of one of the mean branch's workgroups beside these

// (Measured against plans in several rounds that are estimated equal: backward of [128,56,56,64], filter 13, 72.7 us in 252
// workgroups, 80.2 in 428.  The mean branch's count too: forward of [8,112,112,48], filter 17, 17 us with units left for its 8
// workgroups, 21.8 without.  Each of them takes a unit for a whole turn: forward of [32,56,56,64], filter 13, with 32 of them,
// 15.8 us on 224 workgroups, 18.7 on 268 by a share of 5 us each, which left the last 12 a unit only when the convolutions ended.)
// Steps per run with which all problems end together, as early as 256 compute units with one workgroup each allow, the mean
// branch's nmean short workgroups one after another on the units left over; false: they do not fit in one round.
template <int N>
inline bool launch_balance(const LaunchPart (&p)[N], int nmean, int (&steps)[N]) {
    auto fits = [&](double t, int (&s)[N]) {
        const int turns = t < 2 * kMeanCost ? 1 : (int)(t / kMeanCost);   // of a unit, within the launch
        double units = (nmean + turns - 1) / turns;
        for (int i = 0; i < N; ++i) {
            const double most = (t - p[i].start) / p[i].step;
            s[i] = most >= p[i].total ? p[i].total : (int)most;
            if (s[i] < p[i].least) return false;
            units += (double)p[i].blocks(s[i]);
        }
        return units <= 256.0;
    };
    double lo = 0, hi = kMeanCost;
    for (const LaunchPart& q : p) hi = std::max(hi, q.start + q.step * (q.total + 0.5));
    if (!fits(hi, steps)) return false;
    for (int i = 0; i < 24; ++i) {
        const double t = 0.5 * (lo + hi);
        int s[N];
        if (fits(t, s)) hi = t;
        else lo = t;
    }
    return fits(hi, steps);
}

// (a tile of two images starts later)
inline LaunchPart tz_part(const TzGeom& g, int ni, double start, double step) {
    return {start + 1.3 * (ni - 1), step, cdiv(tz_rows(g, ni), 8), 1, [g, ni](int steps) {
                TzGeom c = g;
                return tz_cut_steps(c, ni, steps) ? tz_blocks(c) : 1LL << 40;
            }};
}

// Candidates of a problem of dwconv_tz.h where that does not apply: n is the rows of the runs.
inline void tz_cuts(std::vector<LaunchCut>& out, TzGeom g, int ni, double start, double step) {
    auto add = [&](int steps) {
        if (steps >= 1 && tz_cut_steps(g, ni, steps)) out.push_back({g.run, start + step * tz_steps(g), tz_blocks(g)});
    };
    if (!tz_cut_alone(g, ni)) return;
    const int alone = tz_steps(g);
    for (int e : {1, 2, 4, 8}) add(alone * e);
    add(cdiv(g.OH, 8));
}

struct Fwd2Plan {
    int n[2];     // rows of the runs of the full and of the half scale
    int first;    // problem whose workgroups come first in the grid
};

template <int K, int CS>
static Fwd2Plan fwd2_plan(int B, const TzGeom& g0, int npc0, const TzGeom& g1, int npc1, int nmean) {
    static std::mutex mu;
    struct Key {
        int B, H, W, h, w, C, nmean;
        bool operator<(const Key& o) const {
            return std::tie(B, H, W, h, w, C, nmean) < std::tie(o.B, o.H, o.W, o.h, o.w, o.C, o.nmean);
        }
    };
    static std::map<Key, Fwd2Plan> cache;
    const Key key{B, g0.OH, g0.OW, g1.OH, g1.OW, g0.C, nmean};
    std::lock_guard<std::mutex> lock(mu);
    if (auto it = cache.find(key); it != cache.end()) return it->second;
    Fwd2Plan best{{8, 8}, 0};
    const int ni[2] = {16 / npc0, 16 / npc1};
    const LaunchPart parts[2] = {tz_part(g0, ni[0], kTzStart, kTzStep), tz_part(g1, ni[1], kTzStart, kTzStep)};
    int steps[2];
    if (launch_balance(parts, nmean, steps)) {
        TzGeom c0 = g0, c1 = g1;
        tz_cut_steps(c0, ni[0], steps[0]), tz_cut_steps(c1, ni[1], steps[1]);
        best = Fwd2Plan{{c0.run, c1.run}, 0};
    } else {
        std::vector<LaunchCut> cuts[2];
        tz_cuts(cuts[0], g0, ni[0], kTzStart, kTzStep), tz_cuts(cuts[1], g1, ni[1], kTzStart, kTzStep);
        const LaunchCut mean{0, kMeanCost, nmean};
        double best_t = 0;
        for (const LaunchCut& f : cuts[0])
            for (const LaunchCut& q : cuts[1]) {
                const LaunchCut* const pick[3] = {&f, &q, &mean};
                const int ord[3] = {f.cost >= q.cost ? 0 : 1, f.cost >= q.cost ? 1 : 0, 2};   // longest first
                const double t = launch_makespan(pick, ord);
                if (best_t == 0 || t < best_t - 1e-9) best_t = t, best = Fwd2Plan{{f.n, q.n}, ord[0]};
            }
    }
    if (cache.size() >= kPlanCacheMax) cache.clear();   // callers with ever-changing shapes: a plan is cheap to redo
    cache[key] = best;
    return best;
}

template <typename T, int K, int CS, int NPC0, int NPC1, int MODE>
static void fwd2_go(const Fwd2Args& a, unsigned grid, size_t lds, hipStream_t s) {
    auto kern = dwconv_fwd2_k<T, K, CS, NPC0, NPC1, MODE>;
    static std::once_flag once;
    std::call_once(once, [&] { (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); });
    hipLaunchKernelGGL(kern, dim3(grid), dim3(512), lds, s, a);
}

// -1: not covered (the caller makes the two launches).  16-bit types, C % 8 == 0, padding K / 2; the full scale
// [B, H, W, C], the pooled one [B, h, w, C].
// gate0, gate1 (both or neither, the full scale in the wide tile): the gate in the store of each scale, y0 / y1 then being the gated tensors with the
// strides and channel offsets the gates name.
template <int K>
static int launch_fwd2(const void* x0, const void* w0, void* y0, const void* x1, const void* w1, void* y1, int B, int H,
                       int W, int h, int w, int C, int dtype, hipStream_t s, const TzGate* gate0 = nullptr,
                       const TzGate* gate1 = nullptr, const PoolFwdJob* mean = nullptr) {
    constexpr int CS = (2 * 4 * TzShape<K, 16, 16>::NM + 2 * 4 * TzShape<K, 16, 16>::RING) <= 160 ? 16 : 8;
    if (dtype == kF32 || C % 8 != 0 || B < 1 || H < 1 || W < 1 || h < 1 || w < 1) return -1;
    if ((gate0 != nullptr) != (gate1 != nullptr) || (gate0 && !tz_wide_tile(B, W))) return -1;
    const int P = K / 2;
    for (const void* p : {x0, w0, (const void*)y0, x1, w1, (const void*)y1})
        if (!p || (reinterpret_cast<uintptr_t>(p) & 15)) return -1;
    Fwd2Args a{};
    Fwd2Problem &f = a.p[0], &q = a.p[1];
    f.npc = tz_wide_tile(B, W) ? 16 : 8, q.npc = tz_wide_tile(B, w) ? 16 : 8;
    auto geom = [&](Fwd2Problem& p, int hh, int ww, const TzGate* gate) {
        return p.npc == 16 ? tz_make_geom<K, 16, CS>(p.g, false, B, hh, ww, C, P, P, false, gate)
                           : tz_make_geom<K, 8, CS>(p.g, false, B, hh, ww, C, P, P, false, gate);
    };
    if (!geom(f, H, W, gate0) || !geom(q, h, w, gate1)) return -1;
    Fwd2Plan plan = fwd2_plan<K, CS>(B, f.g, f.npc, q.g, q.npc, mean ? mean->B : 0);
    if (const char* e = tune_env("PDW_FWD2_BANDS")) {   // "rows of the runs of the full scale, of the half scale, first problem"
        if (sscanf(e, "%d,%d,%d", &plan.n[0], &plan.n[1], &plan.first) != 3) return -1;
    }
    if (tune_env("PDW_FWD2_PRINT"))
        fprintf(stderr, "fwd2 plan B=%d H=%d W=%d C=%d K=%d: runs %d %d first %d\n", B, H, W, C, K, plan.n[0], plan.n[1], plan.first);
    long long n[2];
    for (int i = 0; i < 2; ++i) {
        if (!tz_cut(a.p[i].g, 16 / a.p[i].npc, plan.n[i])) return -1;
        n[i] = tz_blocks(a.p[i].g);
    }
    const int nmean = mean ? mean->B : 0;
    if (n[0] + n[1] + nmean > 0x7fffffffLL) return -1;
    a.mean = mean ? *mean : PoolFwdJob{};
    f.x = x0, f.w = w0, f.y = y0, f.n = (int)n[0], f.start = plan.first == 0 ? 0 : (int)n[1];
    q.x = x1, q.w = w1, q.y = y1, q.n = (int)n[1], q.start = plan.first == 0 ? (int)n[0] : 0;
    size_t lds = 0;
    for (const Fwd2Problem& p : a.p) lds = std::max(lds, p.npc == 16 ? TzShape<K, 16, CS>::lds_bytes : TzShape<K, 8, CS>::lds_bytes);
    if (nmean > 0) lds = std::max(lds, (size_t)9 * mean->D * sizeof(float));
    const unsigned grid = (unsigned)(n[0] + n[1] + nmean);
    auto go = [&](auto t, auto mode) {
        using T = decltype(t);
        constexpr int MODE = decltype(mode)::value;
        if constexpr (CS == 16) {
            if (f.npc == 16 && q.npc == 16) return fwd2_go<T, K, CS, 16, 16, MODE>(a, grid, lds, s);
            if (f.npc == 16) return fwd2_go<T, K, CS, 16, 8, MODE>(a, grid, lds, s);
        }
        if constexpr (CS != 16 || MODE == 0) fwd2_go<T, K, CS, 0, 0, MODE>(a, grid, lds, s);
    };
    using Plain = std::integral_constant<int, 0>;
    using Gated = std::integral_constant<int, 4>;
    if (gate0) dtype == kF16 ? go(f16_t{}, Gated{}) : go(bf16_t{}, Gated{});
    else dtype == kF16 ? go(f16_t{}, Plain{}) : go(bf16_t{}, Plain{});
    return check_launch("dwconv_fwd2");
}

}  // namespace pdw
