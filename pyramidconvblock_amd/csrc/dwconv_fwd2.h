// The forward convolutions of both scales of a two-scale block as one launch: y0 = conv(x0, w0) at the full scale and
// y1 = conv(x1, w1) at the pooled one (x1 being the average pool of x0, made before the launch), neither
// depending on the other.  A compute unit holds one workgroup of these kernels at a time and a band costs a start-up
// that does not depend on its height, so a launch of its own cuts a problem into enough bands to fill the chip; here
// the full scale runs as whole-image bands on half of the compute units while the half scale's workgroups run on the
// others (14.8 us against 13.9 + 7.9 us and a launch gap at [32,56,56,64], K = 13).  Each scale runs in the tile
// (16 or 8 patches side by side) that its width fills better: by template where the full scale's is the wide one and slices
// are 16 channels (each workgroup starts with one problem's arguments and no choice between the fields of two; at run time,
// us: filter 13 14.2 for 14.0; [128,56,56,64] filter 13 36.0 for 35.7), at run time elsewhere (with the mean branch, filters
// 15 and 17: 24.7 and 24.6, by template 24.9 and 24.8).
// The kernel template and its per-filter-size launcher; dwconv_fwd2_k<K>.hip instantiate it, one file per size.
#pragma once
#include <algorithm>
#include <map>
#include <queue>
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

// Workgroups dealt in grid order to the earliest free of 256 compute units: the time the last one ends.
inline double tz_makespan(int nproblems, const double* cost, const long long* count, const int* ord) {
    constexpr int kCU = 256;
    std::priority_queue<double, std::vector<double>, std::greater<double>> free_at;
    for (int c = 0; c < kCU; ++c) free_at.push(0.0);
    double end = 0;
    for (int o = 0; o < nproblems; ++o)
        for (long long n = 0; n < count[ord[o]]; ++n) {
            const double t = free_at.top() + cost[ord[o]];
            free_at.pop();
            free_at.push(t);
            end = std::max(end, t);
        }
    return end;
}

struct Fwd2Plan {
    int nb[2];    // bands of the full and of the half scale
    int first;    // problem whose workgroups come first in the grid
};

// Band costs in microseconds fitted to traces at [32,56,56,64]: a 64-column band of one image 9.6 + 0.045 per row
// (K = 13), a 32-column band of two images 3.7 + 0.175 per row.
template <int K, int CS>
inline double tz_band_cost(int npc, int br) {
    const double work = TzShape<K, 16, CS>::NM / 8.0;
    if (npc == 16) return (CS == 16 ? 9.6 : 7.0) + 0.045 * br * work;
    return (CS == 16 ? 3.7 : 3.0) + 0.175 * br * work;
}

template <int K, int CS>
static Fwd2Plan fwd2_plan(int B, const TzGeom& g0, int npc0, const TzGeom& g1, int npc1) {
    static std::mutex mu;
    struct Key {
        int B, H, W, h, w, C;
        bool operator<(const Key& o) const { return std::tie(B, H, W, h, w, C) < std::tie(o.B, o.H, o.W, o.h, o.w, o.C); }
    };
    static std::map<Key, Fwd2Plan> cache;
    const Key key{B, g0.OH, g0.OW, g1.OH, g1.OW, g0.C};
    std::lock_guard<std::mutex> lock(mu);
    if (auto it = cache.find(key); it != cache.end()) return it->second;
    const int oh[2] = {g0.OH, g1.OH}, npc[2] = {npc0, npc1};
    const long long per_band[2] = {(long long)cdiv(B, 16 / npc0) * g0.ncolt * g0.nslices,
                                   (long long)cdiv(B, 16 / npc1) * g1.ncolt * g1.nslices};
    const int standalone[2] = {g0.nbands, g1.nbands};
    Fwd2Plan best{{standalone[0], standalone[1]}, 0};
    double best_t = 0;
    const bool plenty = per_band[0] + per_band[1] > 1536;   // the chip is full whatever the cut: fewest start-ups
    const int cand[4] = {1, 2, 4, 0};                       // 0: the stand-alone planner's count
    for (int a = 0; a < 4; ++a)
        for (int b = 0; b < 4; ++b) {
            if (plenty && (a | b) != 0) continue;
            const int pick[2] = {cand[a], cand[b]};
            int nb[2];
            double cost[2];
            long long count[2];
            bool ok = true;
            for (int i = 0; i < 2; ++i) {
                nb[i] = pick[i] ? pick[i] : standalone[i];
                if (pick[i] && nb[i] > std::max(1, oh[i] / 4)) ok = false;
                const int br = (cdiv(oh[i], nb[i]) + 3) / 4 * 4;
                nb[i] = cdiv(oh[i], br);
                cost[i] = tz_band_cost<K, CS>(npc[i], br), count[i] = per_band[i] * nb[i];
            }
            if (!ok) continue;
            const int ord[2] = {cost[0] >= cost[1] ? 0 : 1, cost[0] >= cost[1] ? 1 : 0};   // longest first
            const double t = plenty ? 1.0 : tz_makespan(2, cost, count, ord);
            if (best_t == 0 || t < best_t - 1e-9) best_t = t, best = Fwd2Plan{{nb[0], nb[1]}, ord[0]};
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
        long long n;
        return p.npc == 16 ? tz_make_geom<K, 16, CS>(p.g, n, false, B, hh, ww, C, P, P, false, gate)
                           : tz_make_geom<K, 8, CS>(p.g, n, false, B, hh, ww, C, P, P, false, gate);
    };
    if (!geom(f, H, W, gate0) || !geom(q, h, w, gate1)) return -1;
    Fwd2Plan plan = fwd2_plan<K, CS>(B, f.g, f.npc, q.g, q.npc);
    if (const char* e = tune_env("PDW_FWD2_BANDS")) {   // "bands of the full scale, of the half scale, first problem"
        if (sscanf(e, "%d,%d,%d", &plan.nb[0], &plan.nb[1], &plan.first) != 3) return -1;
    }
    if (tune_env("PDW_FWD2_PRINT"))
        fprintf(stderr, "fwd2 plan B=%d H=%d W=%d C=%d K=%d: bands %d %d first %d\n", B, H, W, C, K, plan.nb[0], plan.nb[1], plan.first);
    long long n[2];
    for (int i = 0; i < 2; ++i) {
        TzGeom& g = a.p[i].g;
        g.BR = (cdiv(g.OH, plan.nb[i]) + 3) / 4 * 4, g.nbands = cdiv(g.OH, g.BR);
        n[i] = (long long)cdiv(B, 16 / a.p[i].npc) * g.nbands * g.ncolt * g.nslices;
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
