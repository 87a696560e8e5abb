// The three convolution launches at the end of a two-scale block's backward pass that do not depend on one another
// (the full-scale input gradient, with the pooled branch's gradient added where the pool halved the extents, and the weight
// gradients of both scales) as one launch: on a compute unit a band of each runs back to back, without two drains and
// launch gaps in between.  Every problem runs in the tile that its width fills better: by template where the input
// gradient's is the wide one, the pool halved the extents and no mean branch rides along (each workgroup starts with one
// problem's arguments), at run time per problem elsewhere.  (With bands of one image the template was 0.2 to 1.2 us faster; with runs
// both take as long: [32,56,56,64] filter 9 26.0 and 25.9 us, 13 28.6 and 28.7, [128,56,56,64] filter 13 76.0 and 76.5.)
// The kernel template and its per-filter-size launcher; dwconv_bwd3_k<K>.hip instantiate it, one file per size.
#pragma once
#include "dwconv_fwd2.h"
#include "dwconv_tz.h"
#include "dwconv_wgrad_ph.h"
#include <algorithm>
#include <array>
#include <map>
#include <tuple>
#include <type_traits>
#include <vector>

#include "mean_any.h"
#include "reduce_parts.h"

namespace pdw {

struct Bwd3Wgrad {
    const void *x, *gy;
    float* part;
    WgPhGeom g;
    int start, n;  // first workgroup and number of workgroups
};

struct Bwd3Args {
    const void *gy, *w, *add;   // input gradient: dx = conv^T(gy, w) (+ the gradient of a pool of dx's tensor: add / 4 over 2x2 blocks, or by bins)
    void* dx;
    TzGeom gd;
    int npcd;                   // patches of its tile side by side (16 or 8)
    int sd, nd;
    Bwd3Wgrad p[2];          // full scale, pooled scale
    MeanJob mean;               // nmean workgroups behind the others: the backward of the block's mean branch, which needs
    int nmean;                  // nothing of this launch and whose result is read after it
};

template <typename T, int K>
__device__ __forceinline__ void bwd3_wgrad(const void* x, const void* gy, float* part, const WgPhGeom& g, int blk, int nblk) {
    dwconv_wgrad_ph_body<T, wgrad_ph_ncopy(K), wgrad_ph_gr(K)>((const T*)x, (const T*)gy, part, g, blk, nblk);
}

// Each problem's workgroups are a contiguous range of the grid, in the order the launcher chose.
// WIDE: the input gradient's tile is 16 patches, and no mean branch; else as the arguments say.
template <typename T, int K, int CS, bool WIDE, int MODE>
__global__ __launch_bounds__(512, 1) void dwconv_bwd3_k(const Bwd3Args a) {
    const int blk = blockIdx.x;
    if constexpr (WIDE) {
        if ((unsigned)(blk - a.sd) < (unsigned)a.nd)
            dwconv_tz_body<T, K, 16, CS, MODE>((const T*)a.gy, (const T*)a.w, (const T*)a.add, nullptr, (T*)a.dx, a.gd, blk - a.sd, a.nd);
        else if ((unsigned)(blk - a.p[1].start) < (unsigned)a.p[1].n)
            bwd3_wgrad<T, K>(a.p[1].x, a.p[1].gy, a.p[1].part, a.p[1].g, blk - a.p[1].start, a.p[1].n);
        else
            bwd3_wgrad<T, K>(a.p[0].x, a.p[0].gy, a.p[0].part, a.p[0].g, blk - a.p[0].start, a.p[0].n);
    } else {
        if (blk >= a.nd + a.p[0].n + a.p[1].n) {
            extern __shared__ uint32_t smem[];
            mean_bwd_body<T, 512, true>(a.mean, blk - a.nd - a.p[0].n - a.p[1].n, reinterpret_cast<float*>(smem));
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
        const WgPhGeom g = full ? a.p[0].g : a.p[1].g;
        bwd3_wgrad<T, K>(x, gy, part, g, blk - (full ? a.p[0].start : a.p[1].start), full ? a.p[0].n : a.p[1].n);
    }
}

// Cuts and grid order of the three problems.  A compute unit holds one workgroup of this launch at a time, and a workgroup
// costs a start-up (first rows, operand set-up) that does not depend on how many rows it takes, so unlike a launch of its
// own, which has to fill the chip, a problem here is best cut into as few pieces as the other problems leave room for: all
// three in one round of the chip, ending together, where that is possible; else each candidate (runs of several lengths)
// is priced by dealing its workgroups, longest problem first (the grid
// order), to the compute units.  us a call with its two summations, 20 of them in a graph, against whole-image bands of one
// image: [32,56,56,64] filter 9 32.8 -> 25.9, 13 32.3 -> 28.5, 15 43.5 -> 33.9; [128,56,56,64] filter 13 100.5 -> 75.8.  What the runs cost: the two problems that share gy read it at different times, and [32,56,56,64]
// filter 13 fetches and writes 67.3 MB where bands moved 51.6 (48.2 are needed).
struct Bwd3Plan {
    int n[3];         // rows of the input gradient's runs; runs of the full scale's and the half scale's weight gradient
    char order[4];    // 'D', 'F', 'H' in grid order
    bool any_pays;    // the gradient of a pool of other ratios than halves is best added in this launch
};

// Prices of the input gradient here: its store adds the pooled gradient, and its runs have the chip and its memory to share with
// the weight gradients' (256 of them alone: 6.1 + 1.8 a step at filter 13).
constexpr double kBwd3Start = 5.0, kBwd3Step = 1.15;

// Whether the gradient of a pool of other ratios is better added in the input gradient's store (MODE 16) than by avgpool_bwd_k behind the
// launch, which takes 2.8 us and 0.6 a MB of the gradient: a run starts 1 us later and its steps are longer by the bins' loads, which the launch
// waits for as far as its runs are the last to end.  Of 327 random shapes, in the store always, 52 are slower than by two launches, by up to 18 %
// (us, two launches and the store: [3,103,103,600] filter 17 76.6 and 90.6, [107,13,14,640] 93.7 and 110, [54,11,8,664] filter 9 31.1 and 33.6,
// [3,66,65,448] filter 15 31.8 and 34.4); by this rule 4, by 1 % of the step's kernels at most, and the sum of all is 9 % less than by two
// launches.  In the store, as chosen: [3,57,61,200] filter 9 16.7 -> 14.3, [70,57,57,128] filter 7 73.9 -> 54.7, [2,83,82,208] filter 15 20.0 -> 17.1.
template <int K>
static bool bwd3_any_pays(const Bwd3Plan& plan, TzGeom gd, int ni, WgPhPlan p0, WgPhPlan p1, int nmean) {
    constexpr double kAny = K == 3 ? 0.65 : K == 5 ? 0.3 : K == 9 ? 0.7 : K == 15 ? 0.45 : 0.6;   // (us a step; a tenth less, and a few are slower)
    if (!dwconv_bwd3_adds_any(K) || !tz_cut(gd, ni, plan.n[0]) || !wgrad_ph_cut(p0, plan.n[1]) || !wgrad_ph_cut(p1, plan.n[2])) return false;
    auto end = [&](double start, double step) {
        const LaunchCut d{0, start + 1.3 * (ni - 1) + step * tz_steps(gd), tz_blocks(gd)}, mean{0, kMeanCost, nmean};
        const LaunchCut f{0, wgrad_ph_run_cost(K, p0.g.passes), p0.nblocks}, h{0, wgrad_ph_run_cost(K, p1.g.passes), p1.nblocks};
        const LaunchCut* const pick[4] = {&d, &f, &h, &mean};
        int ord[4] = {0, 0, 0, 3};
        for (int i = 0; i < 3; ++i) ord[i] = plan.order[i] == 'D' ? 0 : plan.order[i] == 'F' ? 1 : 2;
        return launch_makespan(pick, ord);
    };
    return end(kBwd3Start + 1.0, kBwd3Step + kAny) - end(kBwd3Start, kBwd3Step) < 2.8 + 0.6 * (2e-6 * gd.B * gd.OH * gd.OW * gd.C);
}

template <int K>
static Bwd3Plan bwd3_plan(int B, const TzGeom& gd, int npcd, const WgPhPlan& p0, const WgPhPlan& p1, int nmean) {
    static std::mutex mu;
    struct Key {
        int B, H, W, h, w, C, nmean;
        bool operator<(const Key& o) const {
            return std::tie(B, H, W, h, w, C, nmean) < std::tie(o.B, o.H, o.W, o.h, o.w, o.C, o.nmean);
        }
    };
    static std::map<Key, Bwd3Plan> cache;
    const Key key{B, gd.OH, gd.OW, p1.g.OH, p1.g.OW, gd.C, nmean};
    std::lock_guard<std::mutex> lock(mu);
    if (auto it = cache.find(key); it != cache.end()) return it->second;
    const int ni = 16 / npcd;
    Bwd3Plan best{{8, 1, 1}, "DFH", false};
    auto part = [](const WgPhPlan& p) { return LaunchPart{kWgPhStart, wgrad_ph_step(K), p.total, p.g.passes, [p](int s) { return p.per_chunk * cdiv(p.total, s); }}; };
    const LaunchPart parts[3] = {tz_part(gd, ni, kBwd3Start, kBwd3Step), part(p0), part(p1)};
    int steps[3];
    if (launch_balance(parts, nmean, steps)) {
        TzGeom c = gd;
        tz_cut_steps(c, ni, steps[0]);
        best = Bwd3Plan{{c.run, cdiv(p0.total, steps[1]), cdiv(p1.total, steps[2])}, "DFH", false};
    } else {
        std::vector<LaunchCut> cuts[3];
        tz_cuts(cuts[0], gd, ni, kBwd3Start, kBwd3Step);
        for (int i = 1; i < 3; ++i) {
            WgPhPlan p = i == 1 ? p0 : p1;
            const int most = p.g.nchunks;
            for (int e = 8; e >= 1; --e) {
                if (!wgrad_ph_cut(p, std::max(1, most * e / 8)) || (!cuts[i].empty() && cuts[i].back().n == p.g.nchunks)) continue;
                cuts[i].push_back({p.g.nchunks, wgrad_ph_run_cost(K, p.g.passes), p.nblocks});
            }
        }
        const LaunchCut mean{0, kMeanCost, nmean};
        double best_t = 0;
        for (const LaunchCut& d : cuts[0])
            for (const LaunchCut& f : cuts[1])
                for (const LaunchCut& q : cuts[2]) {
                    const LaunchCut* const pick[4] = {&d, &f, &q, &mean};
                    int ord[4] = {0, 1, 2, 3};   // (the mean branch's workgroups are the last of the grid)
                    // longest first; the input gradient ahead of a weight gradient of similar length (its run is mostly
                    // start-up, memory latency that overlaps best with the other problems' arithmetic: 29.1 against 30.2 us)
                    auto rank = [&](int x) { return pick[x]->cost * (x == 0 ? 1.25 : 1.0); };
                    std::sort(ord, ord + 3, [&](int x, int y) { return rank(x) > rank(y); });
                    const double t = launch_makespan(pick, ord);
                    if (best_t == 0 || t < best_t - 1e-9) {
                        best_t = t;
                        for (int i = 0; i < 3; ++i) best.n[i] = pick[i]->n, best.order[i] = "DFH"[ord[i]];
                        best.order[3] = 0;
                    }
                }
    }
    best.any_pays = bwd3_any_pays<K>(best, gd, ni, p0, p1, nmean);
    if (cache.size() >= kPlanCacheMax) cache.clear();   // callers with ever-changing shapes: a plan is cheap to redo
    cache[key] = best;
    return best;
}

// The same for the input gradient and the weight gradient of one convolution by itself (no second scale): the cuts that are
// estimated to end first, of one round or several; n[0] = 0 where a launch each is estimated to take no longer.  Together they save a launch and
// fill the rounds that 72 slices, say, leave open (2 x 216 workgroups, or 288 + 216 in two rounds); apart, each side has the chip and its
// memory to itself and its steps are shorter ([64,56,56,128] filter 13 in one round 83.7 us, apart 70.1, [39,45,45,216] filter 17 117
// and 87).  Prices fitted to both of 160 random shapes with cold buffers.  What they do not see: in several rounds, runs of either side longer than
// by itself leave both sides short of memory all the time (with the estimate 0 to 10 % ahead [97,10,11,896] filter 9 64.7 -> 71.6, [75,12,12,624]
// filter 7 42.0 -> 44.8; as long as by itself, 220 such plans 0.98 to 1.5 times as fast), so these have to be estimated further ahead.
// Filters 3 and 5 in one round with runs of the weight gradient more than two and a half times as long as by itself are estimated too short
// ([92,7,7,448] filter 5, three times: 26.6 apart, 28.9 together).
// An estimate less than 6 % ahead is as often behind ([11,64,64,432] filter 7 59.1 and 61.4, [124,8,8,432] filter 5 33.3 and 31.4).
// us with the summation, apart and together:
// [8,64,64,1152] filter 9 84 -> 70, [32,28,28,256] filter 13 33.8 -> 28.8, [2,20,20,64] filter 7 13.2 -> 8.6, [11,74,74,688] filter 9 137 -> 109.
template <int K>
static Bwd3Plan bwd2_plan(const TzGeom& gd, int npcd, const WgPhPlan& p0) {
    static std::mutex mu;
    static std::map<std::array<int, 4>, Bwd3Plan> cache;
    const std::array<int, 4> key{gd.B, gd.OH, gd.OW, gd.C};
    std::lock_guard<std::mutex> lock(mu);
    if (auto it = cache.find(key); it != cache.end()) return it->second;
    // us of a run's start and of its steps in a launch of its own, the input gradient's (filters 15 and 17: 8 channels) and the weight
    // gradient's; their steps side by side, in one round and in several (which are full of either side most of the time); what an
    // estimate of one round has to be ahead by, and one of several with longer runs than by itself (launch_makespan adds its own to all of these)
    constexpr double kStartD = 5.5, kStepD = K <= 9 ? 1.25 : K <= 13 ? 1.4 : 1.2, kStartF = kWgPhStart, kStepF = K <= 9 ? 1.25 : K <= 15 ? 1.8 : 2.5,
                     kLaunch = 2.8, kShareOne = K <= 5 ? 1.15 : K <= 9 ? 1.17 : 1.2, kShareMore = K <= 5 ? 1.15 : K <= 9 ? 1.1 : 1.2, kAhead = 1.06,
                     kAheadLonger = 1.1;
    const int ni = 16 / npcd;
    std::vector<LaunchCut> cuts[2];
    TzGeom g = gd;
    double apart = kLaunch + cdiv(p0.nblocks, 256) * (kStartF + kStepF * p0.g.passes);
    long long alone = 0;   // workgroups of the input gradient by itself
    if (tz_cut_alone(g, ni, K <= 5)) {
        const double steps = tz_alone_cost(tz_blocks(g), tz_steps(g), K <= 5);
        apart += K <= 5 ? kStepD * steps : cdiv(tz_blocks(g), 256) * kStartD + kStepD * (steps - cdiv(tz_blocks(g), 256) * 4.5);
        const int runs = g.nruns;
        alone = tz_blocks(g);
        int last = 0;
        for (int e = 2; e <= 16; ++e) {
            const int most = cdiv(cdiv(tz_rows(gd, ni), 8) * (gd.stack ? 1 : cdiv(gd.B, ni)), std::max(1, runs * e / 8));
            if (most != last && tz_cut_steps(g, ni, most)) cuts[0].push_back({g.run, kStepD * tz_steps(g), tz_blocks(g)});
            last = most;
        }
    }
    WgPhPlan p = p0;
    for (int e = 16; e >= 1; --e) {   // (no more runs than by itself: the workspace is sized for those)
        if (!wgrad_ph_cut(p, std::max(1, p0.g.nchunks * e / 16)) || (!cuts[1].empty() && cuts[1].back().n == p.g.nchunks)) continue;
        cuts[1].push_back({p.g.nchunks, kStepF * p.g.passes, p.nblocks});
    }
    Bwd3Plan best{{0, 1, 0}, "DF", false};
    for (const LaunchCut& dc : cuts[0])
        for (const LaunchCut& fc : cuts[1]) {
            const bool single = dc.count + fc.count <= 256;
            if (K <= 5 && single && fc.count * 5 < p0.nblocks * 2) continue;
            const double share = single ? kShareOne : kShareMore;
            const LaunchCut d{dc.n, kStartD + share * dc.cost, dc.count}, f{fc.n, kStartF + share * fc.cost, fc.count};
            const LaunchCut* const pick[2] = {&d, &f};
            const int ord[2] = {d.cost >= f.cost ? 0 : 1, d.cost >= f.cost ? 1 : 0};
            const bool longer = dc.count < alone || fc.count < p0.nblocks;
            const double t = (single ? kAhead : longer ? kAheadLonger : 1.0) * launch_makespan(pick, ord);
            if (t >= apart) continue;
            apart = t;
            best.n[0] = d.n, best.n[1] = f.n;
            best.order[0] = "DF"[ord[0]], best.order[1] = "DF"[ord[1]];
        }
    if (cache.size() >= kPlanCacheMax) cache.clear();
    cache[key] = best;
    return best;
}

template <typename T, int K, int CS, bool WIDE, int MODE>
static void bwd3_go(const Bwd3Args& a, unsigned grid, size_t lds, hipStream_t s) {
    auto kern = dwconv_bwd3_k<T, K, CS, WIDE, MODE>;
    static std::once_flag once;
    std::call_once(once, [&] { (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); });
    hipLaunchKernelGGL(kern, dim3(grid), dim3(512), lds, s, a);
}

// -1: not covered (the caller makes the three launches).  16-bit types, C % 8 == 0, padding K / 2; the full scale
// [B, H, W, C], the pooled one [B, h, w, C].  addp (optional; H = 2 h and W = 2 w or dwconv_bwd3_adds_any): the pooled branch's gradient.
// x1 = nullptr and h = 0: no pooled scale (a convolution by itself; -1 also where two launches take no longer).  With plan_out and addp of other
// ratios than halves, -1 also where adding it by a launch behind is estimated to take no longer.
template <int K>
static int launch_bwd3(const void* gyf, const void* w0, const void* addp, void* dx, const void* x0, void* dw0, void* ws0,
                       const void* x1, const void* gy1, void* dw1, void* ws1, int B, int H, int W, int h, int w, int C, int dtype,
                       hipStream_t s, int* plan_out, const MeanJob* mean) {
    constexpr int CS = (2 * 4 * TzShape<K, 16, 16>::NM + 2 * 4 * TzShape<K, 16, 16>::RING) <= 160 ? 16 : 8;
    const bool one = h == 0;
    if (dtype == kF32 || C % 8 != 0 || B < 1 || H < 1 || W < 1 || (!one && (h < 1 || w < 1))) return -1;
    const bool any = addp && (H != 2 * h || W != 2 * w);
    if (any && (one || h > H || w > W || !dwconv_bwd3_adds_any(K))) return -1;
    const int P = K / 2;
    if (!plan_out)
        for (const void* p : {gyf, w0, (const void*)dx, x0, (const void*)ws0, one ? x0 : x1, one ? gyf : gy1, (const void*)(one ? ws0 : ws1)})
            if (!p || (reinterpret_cast<uintptr_t>(p) & 15)) return -1;
    if (reinterpret_cast<uintptr_t>(addp) & 15) return -1;
    Bwd3Args a{};
    a.npcd = tz_wide_tile(B, W) ? 16 : 8;
    if (!(a.npcd == 16 ? tz_make_geom<K, 16, CS>(a.gd, true, B, H, W, C, K - 1 - P, K - 1 - P, true, nullptr)
                       : tz_make_geom<K, 8, CS>(a.gd, true, B, H, W, C, K - 1 - P, K - 1 - P, true, nullptr)))
        return -1;
    WgPhPlan p0 = wgrad_ph_plan(B, H, W, C, K, P, P), p1;
    if (!one) p1 = wgrad_ph_plan(B, h, w, C, K, P, P);
    if (!p0.ok || (!one && !p1.ok)) return -1;
    MeanJob job{};
    if (mean) job = *mean, job.shared = mean_shared(job.B, job.D);
    const int nmean = mean ? mean_bwd_workgroups(job) : 0;
    Bwd3Plan plan = one ? bwd2_plan<K>(a.gd, a.npcd, p0) : bwd3_plan<K>(B, a.gd, a.npcd, p0, p1, nmean);
    if (const char* e = tune_env("PDW_BWD3_BANDS")) {   // e.g. "64,31,8,DHF": cuts of D, F, H and the grid order
        if (sscanf(e, "%d,%d,%d,%3s", &plan.n[0], &plan.n[1], &plan.n[2], plan.order) != 4) return -1;
    }
    if (tune_env("PDW_BWD3_PRINT"))
        fprintf(stderr, "bwd3 plan B=%d H=%d W=%d C=%d K=%d: cuts D %d F %d H %d order %s\n", B, H, W, C, K, plan.n[0],
                plan.n[1], plan.n[2], plan.order);
    if (plan_out && any && !plan.any_pays) return -1;
    if (plan.n[0] < 1 || plan.n[1] < 1 || (!one && plan.n[2] < 1)) return -1;
    if (!tz_cut(a.gd, 16 / a.npcd, plan.n[0])) return -1;
    const long long nd = tz_blocks(a.gd);
    int parts[2] = {}, per_image[2] = {};   // partials of the weight gradients, pieces of an image
    for (int i = 0; i < (one ? 1 : 2); ++i) {
        WgPhPlan& p = i == 0 ? p0 : p1;
        if (!wgrad_ph_cut(p, plan.n[1 + i])) return -1;
        parts[i] = p.parts(), per_image[i] = cdiv(p.g.nchunks, cdiv(B, p.g.ni));
        a.p[i].g = p.g, a.p[i].n = (int)p.nblocks;
    }
    const long long grid_all = nd + p0.nblocks + (one ? 0 : p1.nblocks) + nmean;
    if (grid_all > 0x7fffffffLL) return -1;
    if (plan_out) {
        plan_out[0] = cdiv(a.gd.nruns, cdiv(B, 16 / a.npcd)), plan_out[1] = per_image[0], plan_out[2] = per_image[1];
        return 0;
    }
    a.gy = gyf, a.w = w0, a.add = addp, a.dx = dx;
    a.p[0].x = x0, a.p[0].gy = gyf, a.p[0].part = (float*)ws0;
    a.p[1].x = x1, a.p[1].gy = gy1, a.p[1].part = (float*)ws1;
    a.nd = (int)nd, a.nmean = nmean;
    a.mean = job;
    {
        // order of the three problems in the grid: a permutation of D (input gradient), H (half scale), F (full scale)
        const char* ord = plan.order;
        int at = 0;
        for (int i = 0; i < 3 && ord[i]; ++i) {
            if (ord[i] == 'D') a.sd = at, at += a.nd;
            if (ord[i] == 'H') a.p[1].start = at, at += a.p[1].n;
            if (ord[i] == 'F') a.p[0].start = at, at += a.p[0].n;
        }
    }
    if (any) a.gd.AH = h, a.gd.AW = w;
    size_t lds = a.npcd == 16 ? TzShape<K, 16, CS>::lds_bytes : TzShape<K, 8, CS>::lds_bytes;
    if (any) lds = (size_t)(a.npcd == 16 ? TzShape<K, 16, CS>::bins_at : TzShape<K, 8, CS>::bins_at) + 8 * (size_t)H;
    if (lds > 160 * 1024) return -1;
    lds = std::max(lds, WgPhShape<wgrad_ph_ncopy(K), wgrad_ph_gr(K)>::lds_bytes);
    if (nmean) lds = std::max(lds, mean_lds(job.D, 512, job.shared ? kMeanImages : 1));
    const unsigned grid = (unsigned)grid_all;
    auto go = [&](auto t) {
        using T = decltype(t);
        if (!addp) bwd3_go<T, K, CS, false, 0>(a, grid, lds, s);
        else if (any) bwd3_go<T, K, CS, false, dwconv_bwd3_adds_any(K) ? 16 : 0>(a, grid, lds, s);
        else if (a.npcd == 16 && nmean == 0) bwd3_go<T, K, CS, true, 1>(a, grid, lds, s);
        else bwd3_go<T, K, CS, false, 1>(a, grid, lds, s);
    };
    if (dtype == kF16) go(f16_t{});
    else go(bf16_t{});
    if (int e = check_launch("dwconv_bwd3")) return e;
    const int n0 = parts[0], n1 = parts[1];
    if (dtype == kF16) {
        if (int e = wgrad_reduce_launch<f16_t>((const float*)ws0, dw0, n0, K * K * C, s)) return e;
        return one ? 0 : wgrad_reduce_launch<f16_t>((const float*)ws1, dw1, n1, K * K * C, s);
    }
    if (int e = wgrad_reduce_launch<bf16_t>((const float*)ws0, dw0, n0, K * K * C, s)) return e;
    return one ? 0 : wgrad_reduce_launch<bf16_t>((const float*)ws1, dw1, n1, K * K * C, s);
}

}  // namespace pdw
