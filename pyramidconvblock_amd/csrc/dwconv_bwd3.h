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
#include "dwconv_wgrad_ph.h"
#include "dwconv_wgrad_tz.h"
#include <algorithm>
#include <map>
#include <tuple>
#include <type_traits>
#include <vector>

#include "mean_any.h"
#include "reduce_parts.h"

namespace pdw {

// The weight gradient's kernel by filter size: phase-major (dwconv_wgrad_ph.h) up to 15, dwconv_wgrad_tz.h beyond.
constexpr bool bwd3_phases(int K) { return K <= kWgPhMaxK; }
template <int K>
using Bwd3Geom = std::conditional_t<bwd3_phases(K), WgPhGeom, WgTzGeom>;

template <int K>
struct Bwd3Wgrad {
    const void *x, *gy;
    float* part;
    Bwd3Geom<K> g;
    int ncb;       // column blocks of a tile (8 or 5; filters beyond 15)
    int start, n;  // first workgroup and number of workgroups
};

template <int K>
struct Bwd3Args {
    const void *gy, *w, *add;   // input gradient: dx = conv^T(gy, w) (+ add / 4 over 2x2 blocks)
    void* dx;
    TzGeom gd;
    int npcd;                   // patches of its tile side by side (16 or 8)
    int sd, nd;
    Bwd3Wgrad<K> p[2];          // full scale, pooled scale
    MeanJob mean;               // nmean workgroups behind the others: the backward of the block's mean branch, which needs
    int nmean;                  // nothing of this launch and whose result is read after it
};

template <typename T, int K, int NCB>
__device__ __forceinline__ void bwd3_wgrad(const void* x, const void* gy, float* part, const Bwd3Geom<K>& g, int blk, int nblk) {
    if constexpr (bwd3_phases(K))
        dwconv_wgrad_ph_body<T, wgrad_ph_ncopy(K), wgrad_ph_gr(K)>((const T*)x, (const T*)gy, part, g, blk, nblk);
    else
        dwconv_wgrad_tz_body<T, NCB>((const T*)x, (const T*)gy, part, g, blk, nblk);
}

// Each problem's workgroups are a contiguous range of the grid, in the order the launcher chose.
// NCB1: column blocks of the pooled scale's tile (filters beyond 15; else 8), the input gradient's tile being 16 patches, the
// full scale's 8 blocks, and no mean branch; 0: all as the arguments say.
template <typename T, int K, int CS, int NCB1, int MODE>
__global__ __launch_bounds__(512, 1) void dwconv_bwd3_k(const Bwd3Args<K> a) {
    const int blk = blockIdx.x;
    if constexpr (NCB1 != 0) {
        if ((unsigned)(blk - a.sd) < (unsigned)a.nd)
            dwconv_tz_body<T, K, 16, CS, MODE>((const T*)a.gy, (const T*)a.w, (const T*)a.add, nullptr, (T*)a.dx, a.gd, blk - a.sd, a.nd);
        else if ((unsigned)(blk - a.p[1].start) < (unsigned)a.p[1].n)
            bwd3_wgrad<T, K, NCB1>(a.p[1].x, a.p[1].gy, a.p[1].part, a.p[1].g, blk - a.p[1].start, a.p[1].n);
        else
            bwd3_wgrad<T, K, 8>(a.p[0].x, a.p[0].gy, a.p[0].part, a.p[0].g, blk - a.p[0].start, a.p[0].n);
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
        const void *x = full ? a.p[0].x : a.p[1].x, *gy = full ? a.p[0].gy : a.p[1].gy;
        float* const part = full ? a.p[0].part : a.p[1].part;
        const Bwd3Geom<K> g = full ? a.p[0].g : a.p[1].g;
        const int at = blk - (full ? a.p[0].start : a.p[1].start), n = full ? a.p[0].n : a.p[1].n;
        if constexpr (bwd3_phases(K)) {
            bwd3_wgrad<T, K, 8>(x, gy, part, g, at, n);
        } else {
            if ((full ? a.p[0].ncb : a.p[1].ncb) == 8) bwd3_wgrad<T, K, 8>(x, gy, part, g, at, n);
            else bwd3_wgrad<T, K, 5>(x, gy, part, g, at, n);
        }
    }
}

// Cuts and grid order of the three problems.  A compute unit holds one workgroup of this launch at a time, and a workgroup
// costs a start-up (first rows, operand set-up) that does not depend on how many rows it takes, so unlike a launch of its
// own, which has to fill the chip, a problem here is best cut into as few pieces as the other problems leave room for: each
// candidate (bands per image: 1, 2, 4 or the stand-alone planner's number; runs of dwconv_wgrad_ph.h: eighths of the
// stand-alone number) is priced by dealing its workgroups, longest problem first (the grid order), to the earliest free of
// 256 compute units.  Costs in microseconds, fitted to traces of this launch at [32,56,56,64]; beside runs of the phase-major
// weight gradient a band of the input gradient takes a quarter longer than beside bands (it shares the memory with faster
// neighbours): without that factor the plan there had 288 workgroups in two rounds, 33.6 us against 31.0 for 244 in one.
struct Bwd3Cut {
    int n;             // bands per image, or runs
    double cost;       // of a workgroup
    long long count;   // workgroups
};
struct Bwd3Plan {
    int n[3];         // of the input gradient, the full scale's and the half scale's weight gradient
    char order[4];    // 'D', 'F', 'H' in grid order
};

// The time the last of `cuts`' workgroups ends, dealt problem by problem in the order `ord`.
inline double bwd3_makespan(const Bwd3Cut* const (&cuts)[3], const int (&ord)[3]) {
    std::map<double, long long> free_at{{0.0, 256}};   // compute units by the time they are free at
    double end = 0;
    for (int o : ord) {
        const Bwd3Cut& c = *cuts[o];
        std::map<double, long long> busy;
        for (long long left = c.count; left > 0;) {
            if (free_at.empty()) std::swap(free_at, busy);
            const auto first = free_at.begin();
            if (!busy.empty() && busy.begin()->first < first->first) {   // some units of this problem are done before
                for (const auto& [t, n] : busy) free_at[t] += n;
                busy.clear();
                continue;
            }
            const double t = first->first + c.cost;
            const long long n = std::min(left, first->second);
            left -= n, busy[t] += n, end = std::max(end, t);
            if ((first->second -= n) == 0) free_at.erase(first);
        }
        for (const auto& [t, n] : busy) free_at[t] += n;
    }
    return end;
}

template <int K, int CS, typename P>
static Bwd3Plan bwd3_plan(int B, const TzGeom& gd, int npcd, const P& p0, const P& p1) {
    static std::mutex mu;
    struct Key {
        int B, H, W, h, w, C;
        bool operator<(const Key& o) const { return std::tie(B, H, W, h, w, C) < std::tie(o.B, o.H, o.W, o.h, o.w, o.C); }
    };
    static std::map<Key, Bwd3Plan> cache;
    const Key key{B, gd.OH, gd.OW, p1.g.OH, p1.g.OW, gd.C};
    std::lock_guard<std::mutex> lock(mu);
    if (auto it = cache.find(key); it != cache.end()) return it->second;
    std::vector<Bwd3Cut> cuts[3];
    const int oh[3] = {gd.OH, p0.g.OH, p1.g.OH};
    long long per_band[3] = {(long long)cdiv(B, 16 / npcd) * gd.ncolt * gd.nslices, 0, 0};
    int standalone[3] = {gd.nbands, 1, 1};
    auto bands = [&](int i, auto cost_of) {   // candidates of a problem that is cut into bands
        // with many times more whole-image bands than compute units the chip is full whatever the cut: fewest start-ups
        const bool plenty = per_band[i] > 1024;
        for (int pick : {1, 2, 4, 0}) {   // 0: the stand-alone planner's number
            if (plenty && pick != 1) continue;
            int nb = pick ? pick : standalone[i];
            // (a weight gradient's partials must fit the workspace sized for the stand-alone plan)
            if (pick && (nb > std::max(1, oh[i] / 4) || (i > 0 && nb > standalone[i]))) continue;
            const int br = (cdiv(oh[i], nb) + 3) / 4 * 4;
            nb = cdiv(oh[i], br);
            cuts[i].push_back({nb, cost_of(br), per_band[i] * nb});
        }
    };
    bands(0, [&](int br) { return (bwd3_phases(K) ? 1.25 : 1.0) * tz_band_cost<K, CS>(npcd, br); });
    for (int i = 1; i < 3; ++i) {
        P p = i == 1 ? p0 : p1;
        if constexpr (bwd3_phases(K)) {
            const int most = p.g.nchunks;
            for (int e = 8; e >= 1; --e) {
                const int n = std::max(1, most * e / 8);
                if (!wgrad_ph_cut(p, n) || (!cuts[i].empty() && cuts[i].back().n == p.g.nchunks)) continue;
                cuts[i].push_back({p.g.nchunks, wgrad_ph_run_cost(K, p.g.passes), p.nblocks});
            }
        } else {
            per_band[i] = (long long)B * p.g.ncolt * p.g.nslices, standalone[i] = p.g.nbands;
            bands(i, [&](int br) { return 3.0 + 3.0 * (p.ncb == 8 ? 1.0 : 0.9) * ((br + 4) / 4); });
        }
    }
    Bwd3Plan best{{cuts[0].back().n, cuts[1].back().n, cuts[2].back().n}, "DFH"};
    double best_t = 0;
    for (const Bwd3Cut& d : cuts[0])
        for (const Bwd3Cut& f : cuts[1])
            for (const Bwd3Cut& q : cuts[2]) {
                const Bwd3Cut* const pick[3] = {&d, &f, &q};
                int ord[3] = {0, 1, 2};
                // longest first; the input gradient ahead of a weight gradient of similar length (its band is mostly
                // start-up, memory latency that overlaps best with the other problems' arithmetic: 29.1 against 30.2 us)
                auto rank = [&](int x) { return pick[x]->cost * (x == 0 ? 1.25 : 1.0); };
                std::sort(ord, ord + 3, [&](int x, int y) { return rank(x) > rank(y); });
                const double t = bwd3_makespan(pick, ord);
                if (best_t == 0 || t < best_t - 1e-9) {
                    best_t = t;
                    for (int i = 0; i < 3; ++i) best.n[i] = pick[i]->n, best.order[i] = "DFH"[ord[i]];
                    best.order[3] = 0;
                }
            }
    if (cache.size() >= kPlanCacheMax) cache.clear();   // callers with ever-changing shapes: a plan is cheap to redo
    cache[key] = best;
    return best;
}

template <typename T, int K, int CS, int NCB1, int MODE>
static void bwd3_go(const Bwd3Args<K>& a, unsigned grid, size_t lds, hipStream_t s) {
    auto kern = dwconv_bwd3_k<T, K, CS, NCB1, MODE>;
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
    if (dtype == kF32 || C % 8 != 0 || B < 1 || H < 1 || W < 1 || h < 1 || w < 1) return -1;
    if (addp && (H != 2 * h || W != 2 * w)) return -1;
    const int P = K / 2;
    if (!plan_out)
        for (const void* p : {gyf, w0, (const void*)dx, x0, (const void*)ws0, x1, gy1, (const void*)ws1})
            if (!p || (reinterpret_cast<uintptr_t>(p) & 15)) return -1;
    if (reinterpret_cast<uintptr_t>(addp) & 15) return -1;
    Bwd3Args<K> a{};
    long long nd;
    a.npcd = tz_wide_tile(B, W) ? 16 : 8;
    if (!(a.npcd == 16 ? tz_make_geom<K, 16, CS>(a.gd, nd, true, B, H, W, C, K - 1 - P, K - 1 - P, true, nullptr)
                       : tz_make_geom<K, 8, CS>(a.gd, nd, true, B, H, W, C, K - 1 - P, K - 1 - P, true, nullptr)))
        return -1;
    auto plan_of = [&](int hh, int ww) {
        if constexpr (bwd3_phases(K)) return wgrad_ph_plan(B, hh, ww, C, K, P, P);
        else return wgrad_tz_plan(B, hh, ww, C, K, P, P);
    };
    auto p0 = plan_of(H, W), p1 = plan_of(h, w);
    if (!p0.ok || !p1.ok) return -1;
    Bwd3Plan plan = bwd3_plan<K, CS>(B, a.gd, a.npcd, p0, p1);
    if (const char* e = tune_env("PDW_BWD3_BANDS")) {   // e.g. "2,2,1,DHF": cuts of D, F, H and the grid order
        if (sscanf(e, "%d,%d,%d,%3s", &plan.n[0], &plan.n[1], &plan.n[2], plan.order) != 4) return -1;
    }
    if (tune_env("PDW_BWD3_PRINT"))
        fprintf(stderr, "bwd3 plan B=%d H=%d W=%d C=%d K=%d: cuts D %d F %d H %d order %s\n", B, H, W, C, K, plan.n[0],
                plan.n[1], plan.n[2], plan.order);
    if (plan.n[0] < 1 || plan.n[1] < 1 || plan.n[2] < 1) return -1;
    auto rows_of = [](int oh, int nb) { return (cdiv(oh, nb) + 3) / 4 * 4; };
    a.gd.BR = rows_of(a.gd.OH, plan.n[0]), a.gd.nbands = cdiv(a.gd.OH, a.gd.BR);
    nd = (long long)cdiv(B, 16 / a.npcd) * a.gd.nbands * a.gd.ncolt * a.gd.nslices;
    int parts[2], per_image[2];   // partials of the weight gradients, pieces of an image
    for (int i = 0; i < 2; ++i) {
        auto& p = i == 0 ? p0 : p1;
        if constexpr (bwd3_phases(K)) {
            if (!wgrad_ph_cut(p, plan.n[1 + i])) return -1;
            parts[i] = p.parts(), per_image[i] = cdiv(p.g.nchunks, cdiv(B, p.g.ni));
        } else {
            p.g.BR = rows_of(p.g.OH, plan.n[1 + i]), p.g.nbands = cdiv(p.g.OH, p.g.BR);
            p.nblocks = (long long)B * p.g.nslices * p.g.ncolt * p.g.nbands;
            parts[i] = B * p.g.nbands * p.g.ncolt, per_image[i] = p.g.nbands;
            a.p[i].ncb = p.ncb;
        }
        a.p[i].g = p.g, a.p[i].n = (int)p.nblocks;
    }
    const int nmean = mean ? mean->B * mean_slices(mean->D) : 0;
    if (nd + p0.nblocks + p1.nblocks + nmean > 0x7fffffffLL) return -1;
    if (plan_out) {
        plan_out[0] = a.gd.nbands, plan_out[1] = per_image[0], plan_out[2] = per_image[1];
        return 0;
    }
    a.gy = gyf, a.w = w0, a.add = addp, a.dx = dx;
    a.p[0].x = x0, a.p[0].gy = gyf, a.p[0].part = (float*)ws0;
    a.p[1].x = x1, a.p[1].gy = gy1, a.p[1].part = (float*)ws1;
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
    if constexpr (bwd3_phases(K)) {
        lds = std::max(lds, WgPhShape<wgrad_ph_ncopy(K), wgrad_ph_gr(K)>::lds_bytes);
    } else {
        for (const Bwd3Wgrad<K>& p : a.p) lds = std::max(lds, p.ncb == 8 ? WgTzShape<8>::lds_bytes : WgTzShape<5>::lds_bytes);
    }
    if (nmean) lds = std::max(lds, mean_lds(mean->D, 512));
    const unsigned grid = (unsigned)(nd + p0.nblocks + p1.nblocks + nmean);
    auto go = [&](auto t) {
        using T = decltype(t);
        const bool wide = a.npcd == 16 && nmean == 0 && (bwd3_phases(K) || a.p[0].ncb == 8);
        if (!addp) return bwd3_go<T, K, CS, 0, 0>(a, grid, lds, s);
        if (!wide) return bwd3_go<T, K, CS, 0, 1>(a, grid, lds, s);
        if constexpr (!bwd3_phases(K)) {
            if (a.p[1].ncb != 8) return bwd3_go<T, K, CS, 5, 1>(a, grid, lds, s);
        }
        bwd3_go<T, K, CS, 8, 1>(a, grid, lds, s);
    };
    if (dtype == kF16) go(f16_t{});
    else go(bf16_t{});
    if (int e = check_launch("dwconv_bwd3")) return e;
    const int n0 = parts[0], n1 = parts[1];
    if (dtype == kF16) {
        if (int e = wgrad_reduce_launch<f16_t>((const float*)ws0, dw0, n0, K * K * C, s)) return e;
        return wgrad_reduce_launch<f16_t>((const float*)ws1, dw1, n1, K * K * C, s);
    }
    if (int e = wgrad_reduce_launch<bf16_t>((const float*)ws0, dw0, n0, K * K * C, s)) return e;
    return wgrad_reduce_launch<bf16_t>((const float*)ws1, dw1, n1, K * K * C, s);
}

}  // namespace pdw
