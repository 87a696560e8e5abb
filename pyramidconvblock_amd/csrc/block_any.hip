// The two-scale pyramid block of conv_block.py:25-49 (scales 1 and s) on any extents, widths and types that the
// library's kernels cover, as one host call each way: what pdw_convblock_* is for the shapes of its fused launches,
// for every other shape (fp32, odd extents, pooled sizes that are not exact halves, widths beyond 128).  Where
// pdw_convblock_supported, these calls are those.  Everything the backward reads lies in one buffer of the caller, so a
// binding keeps one tensor per pass.  A launch sequence of the library's own entry points, chosen from the arguments.
//
// 16-bit blocks whose inner width I is not a multiple of 8 run on channels padded with zeros: both halves of the
// inner channels are laid out G = I / 2 rounded up to 8 wide, so that the matrix-core convolutions (slices of 8 or 16
// channels), the 128 x 128 dense tiles and the 16-byte gate kernels take them; the vector-ALU kernels that take the
// widths as they are cost two to five times as much ([34,55,55,168], filter 15: 693 us for a training step, 1.14 times
// the channels on the matrix cores 324).  The weights are packed into that layout by one launch per forward, and the summations
// of the weight gradients leave the padding out again.
#include <stdint.h>

#include "../../include/pdw.h"
#include "common.h"
#include "kernels.h"
#include "mean_any.h"

namespace {

using namespace pdw;

size_t up256(size_t b) { return (b + 255) & ~(size_t)255; }

// Hands out 256-byte aligned pieces of a buffer; with a null base it only counts.
struct Carver {
    char* base;
    size_t used = 0;
    void* take(size_t bytes) {
        void* r = base ? base + used : nullptr;
        used += up256(bytes);
        return r;
    }
};

struct Shape {
    int B, H, W, h, w, D, I, K, dtype, es, P;   // I: the inner channels as they are laid out
    int G, Gp;            // width of a gate, and of a half of the inner channels
    long long N, n;       // pixels at full and at the pooled resolution
    bool exact;           // the pooled extents are exact halves
    bool single;          // the fused launches of pdw_convblock_* take it
    bool padded() const { return Gp != G; }
    int gw() const { return padded() ? G : 0; }
};

// Width of a half of the inner channels.  Inner widths that are multiples of 8 run as they are: the convolutions and the
// dense tiles take them, and the padding would cost more than 8-byte instead of 16-byte gates (108 against 101 us for a training step
// at [41,16,17,80]).  Others are padded at any size, since the matrix-core convolutions and shared launches take those only: as
// graphs, unpadded and padded, training [1,8,8,40] filter 3 69.4 and 52.2 us, filter 17 125.9 and 57, [2,20,20,136] filter 9 100 and 58,
// inference [1,8,8,40] filter 3 28.3 and 25.3, [1,40,40,248] filter 5 36.1 and 28.4.  Filters beyond 17 run on the vector ALU both
// ways and are padded where the tensor is large ([1,14,14,40], filter 19: 284 and 332).
int padded_half(long long N, int D, int I, int K, int dtype) {
    const bool as_is = dtype == kF32 || D % 8 != 0 || I % 8 == 0 || (K > 17 && D <= 256 && N * I * K * K < 2000000);
    return as_is ? I / 2 : (I / 2 + 7) / 8 * 8;
}

Shape shape_of(int B, int H, int W, int h, int w, int D, int I, int K, int dtype) {
    const int G = I / 2, Gp = padded_half((long long)B * H * W, D, I, K, dtype);
    Shape s{B, H, W, h, w, D, 2 * Gp, K, dtype, dtype == kF32 ? 4 : 2, H * W, G, Gp, (long long)B * H * W, (long long)B * h * w, false, false};
    s.exact = H == 2 * h && W == 2 * w;
    s.single = s.exact && !s.padded() && pdw_convblock_supported(B, H, W, D, I, K, dtype) != 0;
    return s;
}

bool layer_ok(int K, int NO, int dtype) { return pdw_dense_supported(K, NO, dtype) != 0 || dense_wide_ok(K, NO, dtype); }

__global__ __launch_bounds__(256) void pack_weights_k(const PackArgs g) { pack_weights_body(g, blockIdx.x); }

// The block's inner weights as its kernels read them.
struct Weights {
    const void *up, *out, *dw0, *dw1;
};

// What the forward leaves for the backward, and what only the forward needs.
struct Saved {
    void *a, *c0, *cat, *xp, *c1, *m;
    void *up_p, *out_p, *dw0_p, *dw1_p;   // packed weights (padded widths)
    float* yp;   // (forward only, like xparts and ws, but read by the launch that writes y; a row per image)
    float* xparts;
    void* ws;
    size_t bytes;
};

// The mean branch: column sums, and (backward) the sums per image, in the layout of pdw_pool_branch_*.
size_t mean_workspace(const Shape& s) {
    const ColsumJob j = colsum_plan(nullptr, nullptr, s.B, s.P, s.D, s.es);
    const size_t own = up256((size_t)s.B * j.n * s.D * 4) + (size_t)s.B * s.D * 4, old = pdw_pool_branch_workspace_bytes(s.B, s.P, s.D);
    return own > old ? own : old;
}

// The sums of x live until conv_out, the last launch, writes y: they lie in y itself, so that the buffer kept for the
// backward holds no scratch (a sixteenth of a 16-bit x).  In that buffer only where y is too small, images of a few pixels.
Saved saved_layout(const Shape& s, void* base, void* y) {
    Carver c{(char*)base};
    Saved r{};
    const size_t full = (size_t)s.N * s.I * s.es, half = (size_t)s.n * s.I * s.es;
    r.a = c.take(full), r.c0 = c.take(full), r.cat = c.take(full);
    r.xp = c.take(half), r.c1 = c.take(half);
    r.m = c.take((size_t)s.B * s.D * s.es);
    if (s.padded()) {
        const size_t layer = (size_t)s.I * s.D * s.es, filter = (size_t)s.K * s.K * s.I * s.es;
        r.up_p = c.take(layer), r.out_p = c.take(layer), r.dw0_p = c.take(filter), r.dw1_p = c.take(filter);
    }
    r.yp = (float*)c.take((size_t)s.B * s.D * 4);
    const size_t sums = up256((size_t)((s.N + 31) / 32) * s.D * 4), ws = up256(mean_workspace(s));
    char* scratch = (char*)up256((uintptr_t)y);
    if (sums + ws + 255 > (size_t)s.N * s.D * s.es) scratch = (char*)c.take(sums + ws);
    r.xparts = (float*)scratch, r.ws = scratch + sums;
    r.bytes = c.used;
    return r;
}

struct BwdWork {
    void *dcat, *gcf, *gch, *dxp, *da, *gbias;   // (da lies where dcat was: the gates read that before the convolutions write this)
    float *gparts, *dmean;
    void *ws_po, *ws_pool, *ws_w0, *ws_w1, *ws_pu;
    size_t b_po, b_w0, b_w1, b_pu, bytes;
};

BwdWork bwd_layout(const Shape& s, void* base) {
    Carver c{(char*)base};
    BwdWork r{};
    const size_t full = (size_t)s.N * s.I * s.es, half = (size_t)s.n * s.I * s.es;
    const int pad = s.K / 2;
    r.dcat = r.da = c.take(full), r.gcf = c.take(full);
    r.gch = c.take(half), r.dxp = c.take(half);
    r.gbias = c.take((size_t)2 * s.D * s.es);
    r.gparts = (float*)c.take((size_t)((s.N + 31) / 32) * s.D * 4);
    r.dmean = (float*)c.take((size_t)s.B * s.D * 4);
    r.b_po = up256(pdw_dense_wgrad_workspace_bytes(s.N, s.D, s.I)), r.ws_po = c.take(r.b_po);
    r.ws_pool = c.take(mean_workspace(s));
    r.b_w0 = up256(pdw_dwconv_wgrad_workspace_bytes(s.B, s.H, s.W, s.I, s.K, s.K, 1, 1, pad, pad, 1, 1, s.dtype));
    r.ws_w0 = c.take(r.b_w0);
    r.b_w1 = up256(pdw_dwconv_wgrad_workspace_bytes(s.B, s.h, s.w, s.I, s.K, s.K, 1, 1, pad, pad, 1, 1, s.dtype));
    r.ws_w1 = c.take(r.b_w1);
    r.b_pu = up256(pdw_dense_wgrad_workspace_bytes(s.N, s.I, s.D)), r.ws_pu = c.take(r.b_pu);
    r.bytes = c.used;
    return r;
}

PackArgs pack_args(const Shape& s, const Saved& v, const Weights& w) {
    return PackArgs{(const uint16_t*)w.up, (const uint16_t*)w.out, (const uint16_t*)w.dw0, (const uint16_t*)w.dw1,
                    (uint16_t*)v.up_p,     (uint16_t*)v.out_p,     (uint16_t*)v.dw0_p,     (uint16_t*)v.dw1_p,
                    s.D,                   s.G,                    s.Gp,
                    s.I * s.D / 8,         s.I * s.D / 8,          s.K * s.K * s.I / 8};
}

int pack_weights(const PackArgs& g, hipStream_t stream) {
    hipLaunchKernelGGL(pack_weights_k, dim3(pack_workgroups(g)), dim3(256), 0, stream, g);
    return check_launch("pack_weights");
}

bool rows_whole_tiles(const Shape& s) { return s.P % pdw_dense_colsum_rows() == 0; }

int forward(const Shape& s, const Saved& v, const void* x, const Weights& given, const void* w_pool, const void* b_pool,
            const void* b_out, void* y, void* stream) {
    const hipStream_t st = (hipStream_t)stream;
    const Weights wt = s.padded() ? Weights{v.up_p, v.out_p, v.dw0_p, v.dw1_p} : given;
    const void *const w_up = wt.up, *const w_out = wt.out, *const w_dw0 = wt.dw0, *const w_dw1 = wt.dw1;
    // conv_up reads its weights as they were given where it can, and all four are packed by the launch of the pool
    const PackArgs pack = s.padded() ? pack_args(s, v, given) : PackArgs{};
    bool unpacked = s.padded();
    const int pad = s.K / 2, dt = s.dtype;
    const bool two = s.exact && dt != kF32 && pdw_dwconv_fwd2_supported(s.B, s.H, s.W, s.I, s.K, dt);
    // conv_up, where its kernel can with the sums of x per row tile (for the mean branch) and the 2x2 pool of its result
    const float* parts = nullptr;
    int nparts = 0;
    bool pooled = false, first = false;
    const bool any_mean = mean_any_ok(x, w_pool, v.m, s.D, s.es);
    if (two && !s.padded()) {
        const int r = pdw_dense_fwd_colsum_pool(x, w_up, nullptr, v.a, v.xparts, v.xp, s.B, s.H, s.W, s.D, s.I, dt, stream);
        if (r != 0 && r != 3) return r;
        pooled = r == 0;
    }
    // wide layers and fp32 on exact halves: with the pool, the sums of x and the packing, in place of the pool's launch
    if (!pooled && s.exact && any_mean && !pdw_dense_colsum_supported(s.D, s.I, dt)) {
        ColsumJob sums;
        if (dense_wide_first_plan(&sums, s.N, s.D, s.I, s.B, s.P, dt)) {
            sums.x = x, sums.part = (float*)v.ws;
            const int r = dense_wide_first_launch(x, given.up, v.a, v.xp, s.w, s.N, s.D, s.I, sums, s.padded() ? &pack : nullptr, dt, st);
            if (r != 0 && r != -1) return r;
            if (r == 0) pooled = first = true, unpacked = false, parts = sums.part, nparts = sums.n;
        }
    }
    if (first) {
        // (done)
    } else if (s.padded()) {
        const RowMap map{s.Gp, s.G};
        float* const sums = rows_whole_tiles(s) && pdw_dense_colsum_supported(s.D, s.I, dt) ? v.xparts : nullptr;
        int r = dense_rows_launch(x, given.up, 0, nullptr, nullptr, v.a, s.N, s.D, s.I, s.P, dt, st, sums, nullptr, &map);
        if (r == -1) {
            if (int e = pack_weights(pack, st)) return e;
            unpacked = false;
            r = sums ? pdw_dense_fwd_colsum(x, w_up, 0, nullptr, nullptr, v.a, sums, s.N, s.D, s.I, s.P, dt, stream)
                     : pdw_dense_fwd(x, w_up, 0, nullptr, nullptr, v.a, s.N, s.D, s.I, s.P, dt, stream);
        }
        if (r) return r;
        if (sums) parts = sums, nparts = s.P / pdw_dense_colsum_rows();
    } else if (pooled) {
        parts = v.xparts, nparts = s.P / 32;
    } else if (rows_whole_tiles(s) && pdw_dense_colsum_supported(s.D, s.I, dt)) {
        if (int e = pdw_dense_fwd_colsum(x, w_up, 0, nullptr, nullptr, v.a, v.xparts, s.N, s.D, s.I, s.P, dt, stream)) return e;
        parts = v.xparts, nparts = s.P / pdw_dense_colsum_rows();
    } else if (int e = pdw_dense_fwd(x, w_up, 0, nullptr, nullptr, v.a, s.N, s.D, s.I, s.P, dt, stream)) {
        return e;
    }
    // the pool, with the sums of x where conv_up's kernel did not leave any
    auto pool = [&]() -> int {
        const PackArgs* const with = unpacked ? &pack : nullptr;
        unpacked = false;
        if (parts || !any_mean) return avgpool_with_launch(v.a, v.xp, s.B, s.H, s.W, s.I, s.h, s.w, nullptr, with, dt, st);
        const ColsumJob sums = colsum_plan(x, (float*)v.ws, s.B, s.P, s.D, s.es);
        parts = sums.part, nparts = sums.n;
        return avgpool_with_launch(v.a, v.xp, s.B, s.H, s.W, s.I, s.h, s.w, &sums, with, dt, st);
    };
    // the convolutions of both scales                                                         (conv_block.py:14-17)
    bool convs = false, mean = false;
    if (two) {
        if (!pooled)
            if (int e = pool()) return e;
        int r = 3;
        if (parts) {
            r = pdw_dwconv_fwd2_mean(v.a, w_dw0, v.c0, 0, 0, v.xp, w_dw1, v.c1, 0, 0, s.B, s.H, s.W, s.I, s.K, parts, nparts,
                                     w_pool, b_pool, b_out, v.m, v.yp, s.P, s.D, dt, stream);
            mean = r == 0;
        }
        if (r == 3) r = pdw_dwconv_fwd2(v.a, w_dw0, v.c0, v.xp, w_dw1, v.c1, s.B, s.H, s.W, s.I, s.K, dt, stream);
        if (r != 0 && r != 3) return r;
        convs = r == 0;
        if (!convs)
            if (int e = pdw_dwconv_fwd(v.a, w_dw0, v.c0, s.B, s.H, s.W, s.I, s.K, s.K, 1, 1, pad, pad, 1, 1, dt, stream)) return e;
    } else if ((parts || !any_mean) && !unpacked && !pooled) {
        if (int e = pdw_dwconv_fwd_pool(v.a, w_dw0, v.c0, v.xp, s.B, s.H, s.W, s.I, s.K, s.K, 1, 1, pad, pad, 1, 1, s.h, s.w, dt, stream))
            return e;
    } else {
        if (!pooled)
            if (int e = pool()) return e;
        const int r = dt == kF32 ? dwconv_f32t_pair_launch(v.a, w_dw0, v.c0, s.H, s.W, v.xp, w_dw1, v.c1, s.h, s.w, s.B, s.I, s.K, st)
                                 : dwconv_fwd2_launch(v.a, w_dw0, v.c0, v.xp, w_dw1, v.c1, s.B, s.H, s.W, s.h, s.w, s.I, s.K, dt, st);
        if (r != 0 && r != -1) return r;
        convs = r == 0;
        if (!convs)
            if (int e = pdw_dwconv_fwd(v.a, w_dw0, v.c0, s.B, s.H, s.W, s.I, s.K, s.K, 1, 1, pad, pad, 1, 1, dt, stream)) return e;
    }
    if (!convs)
        if (int e = pdw_dwconv_fwd(v.xp, w_dw1, v.c1, s.B, s.h, s.w, s.I, s.K, s.K, 1, 1, pad, pad, 1, 1, dt, stream)) return e;
    // both gates and the resize into the concatenation, the mean branch's row per image, conv_out (conv_block.py:18-21, 40-49)
    if (mean && !s.padded()) {
        const int r = pdw_dense_fwd_gated(v.c0, v.c1, v.cat, w_out, nullptr, v.yp, y, s.B, s.H, s.W, s.I, s.D, 0, dt, stream);
        if (r != 3) return r;
    }
    bool gates = false;
    if (!mean && parts) {
        const int r = block_mid_fwd_launch(v.c0, v.c1, v.cat, s.B, s.H, s.W, s.h, s.w, s.I, s.I, parts, nparts, w_pool, b_pool,
                                           b_out, v.m, v.yp, s.P, s.D, dt, st, s.gw());
        if (r != 0 && r != -1) return r;
        mean = gates = r == 0;
    }
    if (!mean && parts && any_mean) {
        const MeanJob job{parts, nparts, s.B, s.D, 1.f / (float)s.P, w_pool, b_pool, b_out, v.m, v.yp, nullptr, nullptr};
        if (int e = gate_pair_mean_fwd_launch(v.c0, v.c1, v.cat, s.B, s.H, s.W, s.h, s.w, s.I, s.I, job, dt, st, s.gw())) return e;
        mean = gates = true;
    }
    if (!gates)
        if (int e = gate_pair_fwd_launch(v.c0, v.c1, v.cat, s.B, s.H, s.W, s.h, s.w, s.I, s.I, dt, st, s.gw())) return e;
    if (!mean)
        if (int e = pool_branch_fwd_launch(parts ? nullptr : x, w_pool, b_pool, b_out, v.m, v.yp, (float*)v.ws, s.B, s.P, s.D, dt,
                                           st, parts, nparts))
            return e;
    return pdw_dense_fwd(v.cat, w_out, 0, nullptr, v.yp, y, s.N, s.I, s.D, s.P, dt, stream);
}

int backward(const Shape& s, const Saved& v, const BwdWork& g, const void* gy, const void* x, const Weights& wt,
             const void* w_pool, void* dx, void* gw_up, void* gw_dw0, void* gw_dw1, void* gw_pool, void* gb_pool,
             void* gw_out, void* gb_out, void* stream) {
    const int pad = s.K / 2, dt = s.dtype;
    const void *const w_up = wt.up, *const w_out = wt.out, *const w_dw0 = wt.dw0, *const w_dw1 = wt.dw1;
    const hipStream_t st = (hipStream_t)stream;
    // gradients of the inner weights leave the padding out: the halves of a row of channels, or of conv_up's rows
    const int seg = s.padded() ? s.Gp : 0, val = s.G;
    reduce_defer_compact(seg, val);
    // conv_out: gradient of the concatenation and of the weight, with the sums of gy per row tile where the kernel can
    const bool colsum = rows_whole_tiles(s) && pdw_dense_colsum_supported(s.D, s.I, dt);
    const bool pair_cs = colsum && pdw_dense_bwd_pair_colsum_supported(s.D, s.I, dt);
    float* gparts = nullptr;
    const bool any_mean = mean_any_ok(gy, w_pool, v.m, s.D, s.es);
    ColsumJob sums = colsum_plan(gy, (float*)g.ws_pool, s.B, s.P, s.D, s.es);
    // ... or, where that is faster, by workgroups of their own behind those gradients' (else in the gates' launch, as a part of which they take no time)
    const bool ride = any_mean && dense_wide_sums_ride(sums, s.I, dt);
    bool summed = false;
    if (pair_cs || pdw_dense_bwd_pair_supported(s.D, s.I, dt)) {
        if (pair_cs) gparts = g.gparts;
        if (int e = pdw_dense_bwd_pair(gy, w_out, v.cat, g.dcat, gparts, gw_out, g.ws_po, g.b_po, nullptr, 1, s.N, s.D, s.I, dt, stream))
            return e;
    } else {
        const int both = colsum ? -1 : dense_bwd_both_sums_launch(gy, w_out, v.cat, g.dcat, gw_out, g.ws_po, g.b_po, nullptr, 1, s.N, s.D, s.I, dt, st,
                                                                ride ? &sums : nullptr);
        if (both != 0 && both != -1) return both;
        summed = both == 0 && ride;
        if (colsum) {
            gparts = g.gparts;
            if (int e = pdw_dense_fwd_colsum(gy, w_out, 1, nullptr, nullptr, g.dcat, gparts, s.N, s.D, s.I, 1, dt, stream)) return e;
        } else if (both == -1) {
            if (int e = pdw_dense_fwd(gy, w_out, 1, nullptr, nullptr, g.dcat, s.N, s.D, s.I, 1, dt, stream)) return e;
        }
        if (both == -1)
            if (int e = pdw_dense_wgrad(gy, v.cat, gw_out, g.ws_po, g.b_po, s.N, s.D, s.I, dt, stream)) return e;
    }
    // the gates and the mean branch
    reduce_defer_compact(0, 0);
    void* gb0 = gb_out ? gb_out : g.gbias;
    void* gb1 = gb_pool ? gb_pool : (char*)g.gbias + (size_t)s.D * s.es;
    const int nparts = s.P / pdw_dense_colsum_rows();
    int mid = -1;
    MeanJob mean{};
    bool waiting = false;   // the mean branch's backward still has to run
    if (gparts) {
        mid = block_mid_bwd_launch(g.dcat, v.c0, v.c1, g.gcf, g.gch, s.B, s.H, s.W, s.h, s.w, s.I, s.I, gparts, nparts, v.m, w_pool,
                                   gb0, gb1, gw_pool, g.dmean, (float*)g.ws_pool, s.P, s.D, dt, st, s.gw());
        if (mid != 0 && mid != -1) return mid;
    }
    if (mid == -1 && any_mean && reduce_defer_room() >= 5) {
        float* const gs = (float*)((char*)g.ws_pool + up256((size_t)s.B * sums.n * s.D * 4));
        if (int e = gparts || summed ? gate_pair_bwd_launch(g.dcat, v.c0, v.c1, g.gcf, g.gch, s.B, s.H, s.W, s.h, s.w, s.I, s.I, dt, st, s.gw())
                                     : gate_pair_colsum_bwd_launch(g.dcat, v.c0, v.c1, g.gcf, g.gch, s.B, s.H, s.W, s.h, s.w, s.I, s.I, sums, dt, st, s.gw()))
            return e;
        mean = MeanJob{gparts ? gparts : sums.part, gparts ? nparts : sums.n, s.B, s.D, 1.f / (float)s.P, w_pool, nullptr, nullptr, v.m,
                       nullptr, gs, g.dmean};
        waiting = true;
    } else if (mid == -1) {
        if (int e = pool_branch_bwd_launch(gparts ? nullptr : gy, v.m, w_pool, gb0, gb1, gw_pool, g.dmean, (float*)g.ws_pool, s.B,
                                           s.P, s.D, dt, st, gparts, nparts))
            return e;
        if (int e = gate_pair_bwd_launch(g.dcat, v.c0, v.c1, g.gcf, g.gch, s.B, s.H, s.W, s.h, s.w, s.I, s.I, dt, st, s.gw())) return e;
    }
    // the convolutions: the pooled scale's input gradient, then the rest (one launch where that is covered, the mean branch in it)
    reduce_defer_compact(seg, val);
    // (fp32: that gradient together with both weight gradients and the mean branch's backward, then the full scale's input gradient)
    auto f32_pair = [&](const void* w1, void* dx1) {
        return dt != kF32 ? -1 : dwconv_wgrad_f32t_pair_launch(v.a, g.gcf, gw_dw0, g.ws_w0, s.H, s.W, v.xp, g.gch, gw_dw1, g.ws_w1, s.h, s.w, s.B, s.I,
                                                               s.K, pad, st, waiting ? &mean : nullptr, w1, dx1);
    };
    int pair = f32_pair(w_dw1, g.dxp);
    if (pair != 0 && pair != -1) return pair;
    if (pair == -1)
        if (int e = pdw_dwconv_dgrad(g.gch, w_dw1, g.dxp, s.B, s.h, s.w, s.I, s.K, s.K, 1, 1, pad, pad, 1, 1, dt, stream)) return e;
    auto rest = [&](const void* pooled, int* cuts) {
        return dwconv_bwd3_launch(g.gcf, w_dw0, pooled, g.da, v.a, gw_dw0, g.ws_w0, v.xp, g.gch, gw_dw1, g.ws_w1, s.B, s.H, s.W, s.h, s.w, s.I, s.K, dt,
                                  st, cuts, waiting ? &mean : nullptr);
    };
    // (the pooled gradient is added where the full scale's is stored, or behind)
    bool pool_rides = s.exact;
    int r = -1, cuts[3];
    if (pair == -1) {
        if (!s.exact && s.h <= s.H && s.w <= s.W && dwconv_bwd3_adds_any(s.K)) pool_rides = rest(g.dxp, cuts) == 0;
        r = rest(pool_rides ? g.dxp : nullptr, nullptr);
        if (r == -1 && pool_rides && !s.exact) pool_rides = false, r = rest(nullptr, nullptr);
    }
    if (r != 0 && r != -1) return r;
    if (r == -1 && pair == -1) pair = f32_pair(nullptr, nullptr);
    if (pair != 0 && pair != -1) return pair;
    if (waiting) {
        reduce_defer_compact(0, 0);
        if (int e = r == 0 || pair == 0 ? mean_bwd_defer(mean, gb0, gb1, gw_pool, dt, st) : mean_bwd_launch(mean, gb0, gb1, gw_pool, dt, st)) return e;
        reduce_defer_compact(seg, val);
    }
    if (r == 0) {
        if (!pool_rides)
            if (int e = avgpool_bwd_launch(g.dxp, g.da, s.B, s.H, s.W, s.I, s.h, s.w, 1, dt, st)) return e;
    } else {
        if (pair == -1)
            if (int e = pdw_dwconv_wgrad_pair(v.a, g.gcf, gw_dw0, g.ws_w0, g.b_w0, s.H, s.W, v.xp, g.gch, gw_dw1, g.ws_w1, g.b_w1,
                                              s.h, s.w, s.B, s.I, s.K, dt, stream))
                return e;
        if (int e = pdw_dwconv_dgrad_addpool(g.gcf, w_dw0, g.dxp, g.da, s.B, s.H, s.W, s.I, s.K, s.K, 1, 1, pad, pad, 1, 1, s.h,
                                             s.w, dt, stream))
            return e;
    }
    // conv_up: input gradient (plus the mean branch's per-image term) and weight gradient
    reduce_defer_compact(seg * s.D, val * s.D);
    if (dx && s.P >= 32 && pdw_dense_bwd_pair_supported(s.I, s.D, dt))
        return pdw_dense_bwd_pair(g.da, w_up, x, dx, nullptr, gw_up, g.ws_pu, g.b_pu, g.dmean, s.P, s.N, s.I, s.D, dt, stream);
    if (dx) {
        const int both = dense_bwd_both_launch(g.da, w_up, x, dx, gw_up, g.ws_pu, g.b_pu, g.dmean, s.P, s.N, s.I, s.D, dt, st);
        if (both != -1) return both;
    }
    if (int e = pdw_dense_wgrad(g.da, x, gw_up, g.ws_pu, g.b_pu, s.N, s.I, s.D, dt, stream)) return e;
    if (!dx) return 0;
    // (the summations recorded so far ride in the last kernel of the pass)
    return pdw_dense_fwd_flush(g.da, w_up, 1, nullptr, g.dmean, dx, s.N, s.I, s.D, s.P, dt, stream);
}

}  // namespace

extern "C" {

int pdw_block_supported(int B, int H, int W, int h, int w, int D, int I, int K, int dtype) {
    if (dtype != kF32 && dtype != kF16 && dtype != kBF16) return 0;
    if (B < 1 || H < 1 || W < 1 || h < 1 || w < 1 || K < 1 || !(K & 1) || D < 4 || I < 4 || (I & 1)) return 0;
    if ((long long)B * H * W * (D > I ? D : I) > 0x7fffffffLL) return 0;
    // the pool's bins are found in 32-bit products of the extents (the fused launches, on exact halves, need none)
    if (((long long)H * h >= 0x7fffffffLL || (long long)W * w >= 0x7fffffffLL) &&
        !(H == 2 * h && W == 2 * w && pdw_convblock_supported(B, H, W, D, I, K, dtype)))
        return 0;
    if ((long long)B * h * w * I > 0x7fffffffLL) return 0;
    const int Il = 2 * padded_half((long long)B * H * W, D, I, K, dtype);
    if (Il * (long long)B * H * W > 0x7fffffffLL) return 0;
    return layer_ok(D, Il, dtype) && layer_ok(Il, D, dtype) ? 1 : 0;
}

size_t pdw_block_saved_bytes(int B, int H, int W, int h, int w, int D, int I, int K, int dtype) {
    if (!pdw_block_supported(B, H, W, h, w, D, I, K, dtype)) return 0;
    return saved_layout(shape_of(B, H, W, h, w, D, I, K, dtype), nullptr, nullptr).bytes;
}

int pdw_block_fwd(const void* x, const void* w_up, const void* w_dw0, const void* w_dw1, const void* w_pool,
                  const void* b_pool, const void* w_out, const void* b_out, void* y, void* saved, size_t saved_bytes, int B,
                  int H, int W, int h, int w, int D, int I, int K, int dtype, void* stream) {
    if (!pdw_block_supported(B, H, W, h, w, D, I, K, dtype))
        return set_error("pdw_block_fwd: case not covered (B=%d H=%d W=%d h=%d w=%d D=%d I=%d K=%d dtype=%d)", B, H, W, h, w, D,
                         I, K, dtype), 3;
    for (const void* p : {x, w_up, w_dw0, w_dw1, w_pool, w_out, (const void*)y, (const void*)saved})
        if (!p) return set_error("pdw_block_fwd: null pointer"), 1;
    const Shape s = shape_of(B, H, W, h, w, D, I, K, dtype);
    const Saved v = saved_layout(s, saved, y);
    if (saved_bytes < v.bytes)
        return set_error("pdw_block_fwd: buffer of %zu bytes given, %zu needed", saved_bytes, v.bytes), 1;
    const size_t nx = (size_t)s.N * D * s.es;
    if ((uintptr_t)x < (uintptr_t)y + nx && (uintptr_t)y < (uintptr_t)x + nx)
        return set_error("pdw_block_fwd: y overlaps x (it holds sums of x until it is written)"), 1;
    if (s.single)
        return convblock_fwd_launch(x, w_up, w_dw0, w_dw1, w_pool, b_pool, w_out, b_out, v.a, v.c0, v.xp, v.c1, v.cat, v.m, y,
                                    v.xparts, v.yp, B, H, W, D, I, K, dtype, stream);
    return forward(s, v, x, Weights{w_up, w_out, w_dw0, w_dw1}, w_pool, b_pool, b_out, y, stream);
}

size_t pdw_block_bwd_workspace_bytes(int B, int H, int W, int h, int w, int D, int I, int K, int dtype) {
    if (!pdw_block_supported(B, H, W, h, w, D, I, K, dtype)) return 0;
    const Shape s = shape_of(B, H, W, h, w, D, I, K, dtype);
    return bwd_layout(s, nullptr).bytes;
}

int pdw_block_bwd(const void* gy, const void* x, const void* saved, const void* w_up, const void* w_dw0, const void* w_dw1,
                  const void* w_pool, const void* w_out, void* dx, void* gw_up, void* gw_dw0, void* gw_dw1, void* gw_pool,
                  void* gb_pool, void* gw_out, void* gb_out, void* workspace, size_t workspace_bytes, int B, int H, int W,
                  int h, int w, int D, int I, int K, int dtype, void* stream) {
    if (!pdw_block_supported(B, H, W, h, w, D, I, K, dtype))
        return set_error("pdw_block_bwd: case not covered (B=%d H=%d W=%d h=%d w=%d D=%d I=%d K=%d dtype=%d)", B, H, W, h, w, D,
                         I, K, dtype), 3;
    for (const void* p : {gy, x, saved, w_up, w_dw0, w_dw1, w_pool, w_out, (const void*)gw_up, (const void*)gw_dw0,
                          (const void*)gw_dw1, (const void*)gw_pool, (const void*)gw_out, (const void*)workspace})
        if (!p) return set_error("pdw_block_bwd: null pointer"), 1;
    const Shape s = shape_of(B, H, W, h, w, D, I, K, dtype);
    const Saved v = saved_layout(s, const_cast<void*>(saved), nullptr);   // (none of the forward's scratch is read)
    const BwdWork g = bwd_layout(s, workspace);
    if (workspace_bytes < g.bytes)
        return set_error("pdw_block_bwd: workspace of %zu bytes given, %zu needed", workspace_bytes, g.bytes), 1;
    // the final summations of all weight gradients run as one launch at the end of the pass
    if (int e = pdw_reduce_defer_begin()) return e;
    const Weights wt = s.padded() ? Weights{v.up_p, v.out_p, v.dw0_p, v.dw1_p} : Weights{w_up, w_out, w_dw0, w_dw1};
    const int e = backward(s, v, g, gy, x, wt, w_pool, dx, gw_up, gw_dw0, gw_dw1, gw_pool, gb_pool, gw_out, gb_out, stream);
    const int f = pdw_reduce_defer_flush(stream);   // also ends the deferral after an error
    return e ? e : f;
}

}  // extern "C"
