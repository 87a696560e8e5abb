// The three convolution launches at the end of a two-scale block's backward pass that do not depend on one another
// (the full-scale input gradient, with the pooled branch's gradient added where the pool halved the extents, and the weight
// gradients of both scales) as one launch: on a compute unit a band of each runs back to back, without two drains and
// launch gaps in between.  Every problem runs in the tile that its width fills better: by template where both full-scale
// problems' are the wide ones, the pool halved the extents and no mean branch rides along (each workgroup starts with one
// problem's arguments; chosen at run time as for the others, us: [32,56,56,64] filter 13 30.8 for 30.6, 9 32.4 for 31.6,
// 17 50.1 for 49.6; [128,56,56,64] filter 13 98.8 for 97.6), at run time per problem elsewhere.
// The kernel template and its per-filter-size launcher; dwconv_bwd3_k<K>.hip instantiate it, one file per size.
#pragma once
#include "dwconv_fwd2.h"
#include "dwconv_tz.h"
#include "dwconv_wgrad_tz.h"
#include <algorithm>
#include <map>
#include <queue>
#include <tuple>
#include <vector>

#include "mean_any.h"
#include "reduce_parts.h"

namespace pdw {

struct Bwd3Wgrad {
    const void *x, *gy;
    float* part;
    WgTzGeom g;
    int ncb;       // column blocks of a tile (8 or 5)
    int start, n;  // first workgroup and number of workgroups
};

struct Bwd3Args {
    const void *gy, *w, *add;   // input gradient: dx = conv^T(gy, w) (+ add / 4 over 2x2 blocks)
    void* dx;
    TzGeom gd;
    int npcd;                   // patches of its tile side by side (16 or 8)
    int sd, nd;
    Bwd3Wgrad p[2];             // full scale, pooled scale
    MeanJob mean;               // nmean workgroups behind the others: the backward of the block's mean branch, which needs
    int nmean;                  // nothing of this launch and whose result is read after it
};

// Each problem's workgroups are a contiguous range of the grid, in the order the launcher chose.
// NCB1: column blocks of the pooled scale's tile, those of the full scale being 16 patches and 8 blocks, and no mean branch;
// 0: all as the arguments say.
template <typename T, int K, int CS, int NGA, int NCB1, int NB, int MODE>
__global__ __launch_bounds__(512, 1) void dwconv_bwd3_k(const Bwd3Args a) {
    const int blk = blockIdx.x;
    if constexpr (NCB1 != 0) {
        if ((unsigned)(blk - a.sd) < (unsigned)a.nd)
            dwconv_tz_body<T, K, 16, CS, MODE>((const T*)a.gy, (const T*)a.w, (const T*)a.add, nullptr, (T*)a.dx, a.gd, blk - a.sd, a.nd);
        else if ((unsigned)(blk - a.p[1].start) < (unsigned)a.p[1].n)
            dwconv_wgrad_tz_body<T, NGA, NCB1, NB>((const T*)a.p[1].x, (const T*)a.p[1].gy, a.p[1].part, a.p[1].g,
                                                   blk - a.p[1].start, a.p[1].n);
        else
            dwconv_wgrad_tz_body<T, NGA, 8, NB>((const T*)a.p[0].x, (const T*)a.p[0].gy, a.p[0].part, a.p[0].g,
                                                blk - a.p[0].start, a.p[0].n);
    } else {
        if (blk >= a.nd + a.p[0].n + a.p[1].n) {
            extern __shared__ uint32_t smem[];
            mean_bwd_body<T, 512>(a.mean, blk - a.nd - a.p[0].n - a.p[1].n, reinterpret_cast<float*>(smem));
            return;
        }
        if ((unsigned)(blk - a.sd) < (unsigned)a.nd) {
            const T *gy = (const T*)a.gy, *w = (const T*)a.w, *add = (const T*)a.add;
            if (a.npcd == 16) dwconv_tz_body<T, K, 16, CS, MODE>(gy, w, add, nullptr, (T*)a.dx, a.gd, blk - a.sd, a.nd);
            else dwconv_tz_body<T, K, 8, CS, MODE>(gy, w, add, nullptr, (T*)a.dx, a.gd, blk - a.sd, a.nd);
            return;
        }
        const bool full = (unsigned)(blk - a.p[0].start) < (unsigned)a.p[0].n;
        const T *x = (const T*)(full ? a.p[0].x : a.p[1].x), *gy = (const T*)(full ? a.p[0].gy : a.p[1].gy);
        float* const part = full ? a.p[0].part : a.p[1].part;
        const WgTzGeom g = full ? a.p[0].g : a.p[1].g;
        const int at = blk - (full ? a.p[0].start : a.p[1].start), n = full ? a.p[0].n : a.p[1].n;
        if ((full ? a.p[0].ncb : a.p[1].ncb) == 8) dwconv_wgrad_tz_body<T, NGA, 8, NB>(x, gy, part, g, at, n);
        else dwconv_wgrad_tz_body<T, NGA, 5, NB>(x, gy, part, g, at, n);
    }
}

// Band heights and grid order of the three problems.  A compute unit holds one workgroup of this launch at a time, and a
// band costs a start-up (first windows, operand set-up) that does not depend on its height, so unlike a launch of its
// own, which has to fill the chip, a problem here is best cut into as few bands as the other problems leave room for:
// each candidate (1, 2, 4 or the stand-alone planner's number of bands per problem) is priced by dealing its
// workgroups, longest problem first (the grid order), to the earliest free of 256 compute units.  Band costs in
// microseconds, fitted to traces of this launch at [32,56,56,64] (whole-image bands for all three: 28.7 us against
// 37.4 us with the bands of the separate launches at K = 13, 30.3 against 38.5 at K = 9, 50.0 against 60.2 at K = 17).
struct Bwd3Plan {
    int nb[3];        // bands of the input gradient, the full scale's and the half scale's weight gradient
    char order[4];    // 'D', 'F', 'H' in grid order
};

inline double bwd3_makespan(const double (&cost)[3], const long long (&count)[3], const int (&ord)[3]) {
    constexpr int kCU = 256;
    std::priority_queue<double, std::vector<double>, std::greater<double>> free_at;   // earliest free unit on top
    for (int c = 0; c < kCU; ++c) free_at.push(0.0);
    double end = 0;
    for (int o = 0; o < 3; ++o)
        for (long long n = 0; n < count[ord[o]]; ++n) {
            const double t = free_at.top() + cost[ord[o]];
            free_at.pop();
            free_at.push(t);
            end = std::max(end, t);
        }
    return end;
}

template <int K, int CS>
static Bwd3Plan bwd3_plan(int B, const TzGeom& gd, int npcd, const WgTzPlan& p0, const WgTzPlan& p1) {
    static std::mutex mu;
    struct Key {
        int B, H, W, h, w, C;
        bool operator<(const Key& o) const { return std::tie(B, H, W, h, w, C) < std::tie(o.B, o.H, o.W, o.h, o.w, o.C); }
    };
    static std::map<Key, Bwd3Plan> cache;
    const Key key{B, gd.OH, gd.OW, p1.g.OH, p1.g.OW, gd.C};
    std::lock_guard<std::mutex> lock(mu);
    if (auto it = cache.find(key); it != cache.end()) return it->second;
    const int oh[3] = {gd.OH, p0.g.OH, p1.g.OH};
    const long long per_band[3] = {(long long)cdiv(B, 16 / npcd) * gd.ncolt * gd.nslices,
                                   (long long)B * p0.g.ncolt * p0.g.nslices, (long long)B * p1.g.ncolt * p1.g.nslices};
    const int standalone[3] = {gd.nbands, p0.g.nbands, p1.g.nbands};
    constexpr int nmf = K == 17 ? 2 : 1;
    auto band_rows = [&](int i, int nb) { return (cdiv(oh[i], nb) + 3) / 4 * 4; };
    auto band_cost = [&](int i, int br) {
        if (i == 0) return tz_band_cost<K, CS>(npcd, br);
        const int ncb = i == 1 ? p0.ncb : p1.ncb;
        return 3.0 + 1.5 * nmf * (ncb == 8 ? 1.0 : 0.9) * ((br + 4) / 4);
    };
    // the fallback when no candidate survives: every problem cut as its stand-alone launch cuts it
    Bwd3Plan best{{std::max(1, standalone[0]), std::max(1, standalone[1]), std::max(1, standalone[2])}, "DFH"};
    double best_t = 0;
    // with many times more whole-image bands than compute units the chip is full whatever the cut: fewest start-ups
    const bool plenty = per_band[0] + per_band[1] + per_band[2] > 1536;
    const int cand[4] = {1, 2, 4, 0};   // 0: the stand-alone planner's count
    for (int a = 0; a < 4; ++a)
        for (int b = 0; b < 4; ++b)
            for (int c = 0; c < 4; ++c) {
                const int pick[3] = {cand[a], cand[b], cand[c]};
                if (plenty && (a | b | c) != 0) continue;
                int nb[3];
                double cost[3];
                long long count[3];
                bool ok = true;
                for (int i = 0; i < 3; ++i) {
                    nb[i] = pick[i] ? pick[i] : standalone[i];
                    // a weight gradient's partials must fit the workspace sized for the stand-alone plan
                    if (pick[i] && (nb[i] > std::max(1, oh[i] / 4) || (i > 0 && nb[i] > standalone[i]))) ok = false;
                    const int br = band_rows(i, nb[i]);
                    nb[i] = cdiv(oh[i], br);
                    cost[i] = band_cost(i, br), count[i] = per_band[i] * nb[i];
                }
                if (!ok) continue;
                int ord[3] = {0, 1, 2};
                // longest first; the input gradient ahead of a weight gradient of similar length (its band is mostly
                // start-up, memory latency that overlaps best with the other problems' arithmetic: 29.1 against 30.2 us)
                auto rank = [&](int x) { return cost[x] * (x == 0 ? 1.25 : 1.0); };
                std::sort(ord, ord + 3, [&](int x, int y) { return rank(x) > rank(y); });
                const double t = plenty ? 1.0 : bwd3_makespan(cost, count, ord);
                if (best_t == 0 || t < best_t - 1e-9) {
                    best_t = t;
                    for (int i = 0; i < 3; ++i) best.nb[i] = nb[i], best.order[i] = "DFH"[ord[i]];
                    best.order[3] = 0;
                }
            }
    if (cache.size() >= kPlanCacheMax) cache.clear();   // callers with ever-changing shapes: a plan is cheap to redo
    cache[key] = best;
    return best;
}

template <typename T, int K, int CS, int NGA, int NCB1, int NB, int MODE>
static void bwd3_go(const Bwd3Args& a, unsigned grid, size_t lds, hipStream_t s) {
    auto kern = dwconv_bwd3_k<T, K, CS, NGA, NCB1, NB, MODE>;
    static std::once_flag once;
    std::call_once(once, [&] { (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); });
    hipLaunchKernelGGL(kern, dim3(grid), dim3(512), lds, s, a);
}

// -1: not covered (the caller makes the three launches).  16-bit types, C % 8 == 0, padding K / 2; the full scale
// [B, H, W, C], the pooled one [B, h, w, C].  addp (optional, H = 2 h and W = 2 w): the pooled branch's gradient.
template <int K>
static int launch_bwd3(const void* gyf, const void* w0, const void* addp, void* dx, const void* x0, void* dw0, void* ws0,
                       const void* x1, const void* gy1, void* dw1, void* ws1, int B, int H, int W, int h, int w, int C, int dtype,
                       hipStream_t s, int* plan_out, const MeanJob* mean) {
    constexpr int CS = (2 * 4 * TzShape<K, 16, 16>::NM + 2 * 4 * TzShape<K, 16, 16>::RING) <= 160 ? 16 : 8;
    constexpr int NGA0 = (4 + 2 * ((K - 1) / 2) + 3) / 4, NGA = NGA0 < 2 ? 2 : NGA0, NB = K == 17 ? 3 : 2;
    if (dtype == kF32 || C % 8 != 0 || B < 1 || H < 1 || W < 1 || h < 1 || w < 1) return -1;
    if (addp && (H != 2 * h || W != 2 * w)) return -1;
    const int P = K / 2;
    if (!plan_out)
        for (const void* p : {gyf, w0, (const void*)dx, x0, (const void*)ws0, x1, gy1, (const void*)ws1})
            if (!p || (reinterpret_cast<uintptr_t>(p) & 15)) return -1;
    if (reinterpret_cast<uintptr_t>(addp) & 15) return -1;
    Bwd3Args a{};
    long long nd;
    a.npcd = tz_wide_tile(B, W) ? 16 : 8;
    if (!(a.npcd == 16 ? tz_make_geom<K, 16, CS>(a.gd, nd, true, B, H, W, C, K - 1 - P, K - 1 - P, true, nullptr)
                       : tz_make_geom<K, 8, CS>(a.gd, nd, true, B, H, W, C, K - 1 - P, K - 1 - P, true, nullptr)))
        return -1;
    WgTzPlan p0 = wgrad_tz_plan(B, H, W, C, K, P, P), p1 = wgrad_tz_plan(B, h, w, C, K, P, P);
    if (!p0.ok || !p1.ok) return -1;
    Bwd3Plan plan = bwd3_plan<K, CS>(B, a.gd, a.npcd, p0, p1);
    if (const char* e = tune_env("PDW_BWD3_BANDS")) {   // e.g. "2,2,1,DHF": bands of D, F, H and the grid order
        if (sscanf(e, "%d,%d,%d,%3s", &plan.nb[0], &plan.nb[1], &plan.nb[2], plan.order) != 4) return -1;
    }
    if (tune_env("PDW_BWD3_PRINT"))
        fprintf(stderr, "bwd3 plan B=%d H=%d W=%d C=%d K=%d: bands D %d F %d H %d order %s\n", B, H, W, C, K, plan.nb[0],
                plan.nb[1], plan.nb[2], plan.order);
    if (plan.nb[0] < 1 || plan.nb[1] < 1 || plan.nb[2] < 1) return -1;
    auto rows_of = [](int oh, int nb) { return (cdiv(oh, nb) + 3) / 4 * 4; };
    a.gd.BR = rows_of(a.gd.OH, plan.nb[0]), a.gd.nbands = cdiv(a.gd.OH, a.gd.BR);
    nd = (long long)cdiv(B, 16 / a.npcd) * a.gd.nbands * a.gd.ncolt * a.gd.nslices;
    p0.g.BR = rows_of(p0.g.OH, plan.nb[1]), p0.g.nbands = cdiv(p0.g.OH, p0.g.BR);
    p0.nblocks = (long long)B * p0.g.nslices * p0.g.ncolt * p0.g.nbands;
    p1.g.BR = rows_of(p1.g.OH, plan.nb[2]), p1.g.nbands = cdiv(p1.g.OH, p1.g.BR);
    p1.nblocks = (long long)B * p1.g.nslices * p1.g.ncolt * p1.g.nbands;
    if (wgrad_tz_nga(K) != NGA) return -1;
    const int nmean = mean ? mean->B * mean_slices(mean->D) : 0;
    if (nd + p0.nblocks + p1.nblocks + nmean > 0x7fffffffLL) return -1;
    if (plan_out) {
        plan_out[0] = a.gd.nbands, plan_out[1] = p0.g.nbands, plan_out[2] = p1.g.nbands;
        return 0;
    }
    a.gy = gyf, a.w = w0, a.add = addp, a.dx = dx;
    a.p[0] = Bwd3Wgrad{x0, gyf, (float*)ws0, p0.g, p0.ncb, 0, (int)p0.nblocks};
    a.p[1] = Bwd3Wgrad{x1, gy1, (float*)ws1, p1.g, p1.ncb, 0, (int)p1.nblocks};
    a.nd = (int)nd, a.nmean = nmean;
    if (mean) a.mean = *mean;
    {
        // order of the three problems in the grid: a permutation of D (input gradient), H (half scale), F (full scale)
        const char* ord = plan.order;
        int at = 0;
        for (int i = 0; i < 3; ++i) {
            if (ord[i] == 'D') a.sd = at, at += a.nd;
            if (ord[i] == 'H') a.p[1].start = at, at += a.p[1].n;
            if (ord[i] == 'F') a.p[0].start = at, at += a.p[0].n;
        }
    }
    size_t lds = a.npcd == 16 ? TzShape<K, 16, CS>::lds_bytes : TzShape<K, 8, CS>::lds_bytes;
    for (const Bwd3Wgrad& p : a.p) lds = std::max(lds, p.ncb == 8 ? WgTzShape<NGA, 8, NB>::lds_bytes : WgTzShape<NGA, 5, NB>::lds_bytes);
    if (nmean) lds = std::max(lds, mean_lds(mean->D, 512));
    const unsigned grid = (unsigned)(nd + p0.nblocks + p1.nblocks + nmean);
    const bool wide = a.npcd == 16 && p0.ncb == 8 && nmean == 0;
    auto go = [&](auto t) {
        using T = decltype(t);
        if (!addp) bwd3_go<T, K, CS, NGA, 0, NB, 0>(a, grid, lds, s);
        else if (!wide) bwd3_go<T, K, CS, NGA, 0, NB, 1>(a, grid, lds, s);
        else if (p1.ncb == 8) bwd3_go<T, K, CS, NGA, 8, NB, 1>(a, grid, lds, s);
        else bwd3_go<T, K, CS, NGA, 5, NB, 1>(a, grid, lds, s);
    };
    if (dtype == kF16) go(f16_t{});
    else go(bf16_t{});
    if (int e = check_launch("dwconv_bwd3")) return e;
    const int n0 = B * p0.g.nbands * p0.g.ncolt, n1 = B * p1.g.nbands * p1.g.ncolt;
    if (dtype == kF16) {
        if (int e = wgrad_reduce_launch<f16_t>((const float*)ws0, dw0, n0, K * K * C, s)) return e;
        return wgrad_reduce_launch<f16_t>((const float*)ws1, dw1, n1, K * K * C, s);
    }
    if (int e = wgrad_reduce_launch<bf16_t>((const float*)ws0, dw0, n0, K * K * C, s)) return e;
    return wgrad_reduce_launch<bf16_t>((const float*)ws1, dw1, n1, K * K * C, s);
}

}  // namespace pdw
