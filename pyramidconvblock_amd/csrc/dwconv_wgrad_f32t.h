// Depthwise weight gradient in fp32 on the fp32 matrix cores: stride 1, dilation 1, odd square filters 3 .. 17.
//
// With u = 2a + du, v = 8b + dv:  dw[2a+du][8b+dv] = sum over p of xw[p + (2a,8b)] gy[p - (du,dv)],
// one v_mfma_f32_16x16x4_f32 with m = (a,b), n = (du,dv), k = 4 positions: an accumulator of 4 registers holds all taps of a
// channel (filter 17: 27 (a,b), two instructions that share the gy operand).  Four instructions take 16 positions of a row:
// position 4g + t of the block for lane group g in instruction t, so that a lane's four xw values are one aligned
// 16-byte LDS read, and its four gy values two 8-byte pairs at any element offset.
//
// What bounds it: the matrix pipe (32 cycles an instruction; its operands cost the LDS half of that), and next to it the vector
// instructions of the staging, which do not overlap with fp32 products (dwconv_f32t.h): a tick has about 45 of them for 64
// products (157 with every offset and ring row computed per thread).  Every position of a
// row block costs the same whatever the filter, and a row block computes 16 positions of which 8 per tile are margin.
//
// A workgroup (8 wavefronts, one channel each) takes `U` units (image, row band, column tile) of one 8-channel slice one
// after the other as one stream: a tick brings four window rows of x and four rows of gy into LDS rings (requested two
// ticks ahead, across units as well) while the previous ones are multiplied, so only the first unit of a workgroup waits
// for memory.  The taps leave through LDS as 16-byte stores into the workgroup's partial; fixed-order summation, no atomics;
// every four ticks the accumulators are added to a total, so that the error does not grow with a workgroup's share ([32,56,56,64]
// filter 13, against 64 bits: 2.6e-7 of the norm; 4.7e-7 without, 3.5e-7 in halves of an image without).
//
// Measured with the summation (us, before the waits by buffer name, the scalar offsets and the plan below -> with them):
// [32,56,56,64] filter 13 52.7 -> 42.2 (products alone 29; vector ALU, dwconv_wgrad_tiled.h, 78), [3,57,61,100] filter 15 26.9 ->
// 17.9, [8,112,112,48] filter 17 78 -> 63.8, [4,64,64,576] filter 13 110.6 -> 92.2, [100,14,14,64] filter 15 40.9 -> 29.6,
// [6,90,90,32] filter 17 55.8 -> 30.9.  16 channels a workgroup for whole 64-byte requests measured the same.
#pragma once
#include <mutex>

#include "common.h"
#include "dwconv_f32t.h"
#include "kernels.h"
#include "mean_any.h"
#include "tile_common.h"

namespace pdw {

constexpr int wg_f32t_gpitch(int nbi, int ni) {   // gy row pitch: the two rows (du) that a read takes together on other banks
    int p = 4 * ni * (16 * nbi + 8);
    while (p % 256 < 80 || p % 256 > 176) p += 16;
    return p;
}
constexpr int wg_f32t_plane(int bytes) {   // channel quads of a staging write on other banks
    while (bytes % 64 != 32) bytes += 16;
    return bytes;
}
// LDS bytes of a channel: window rows (a ring), gy rows (a ring of nine: the row before the group's four, the next group's)
constexpr int wg_f32t_chx(int K, int nbi, int ni) {
    return wg_f32t_plane(4 * ((4 + 2 * ((K + 1) / 2 - 1) + 3) / 4 + 1) * 4 * ni * (16 * nbi + 8 * ((K + 7) / 8 - 1)));
}
constexpr int wg_f32t_chg(int nbi, int ni) { return wg_f32t_plane(9 * wg_f32t_gpitch(nbi, ni)); }

// NBI 16-column blocks an image (a tile of 16 NBI - 8 columns), NI images side by side; CS channels, a wavefront each.
template <int K, int NBI, int NI>
struct WgF32Shape {
    static constexpr int CS = 8, NT = 64 * CS, NQ = CS / 4;                      // threads; 16-byte pieces of a pixel
    static constexpr int NAU = (K + 1) / 2, NBV = (K + 7) / 8, COMB = NAU * NBV, NMF = (COMB + 15) / 16;
    static constexpr int AM = 2 * (NAU - 1), XG = (4 + AM + 3) / 4;     // groups of four window rows a step reads
    static constexpr int TW = 16 * NBI - 8;                              // gy columns of a tile
    static constexpr int XCI = 16 * NBI + 8 * (NBV - 1), XC = NI * XCI;  // window columns of an image, of all
    static constexpr int RPX = 4 * XC, NRX = 4 * (XG + 1);
    static constexpr int GCI = 16 * NBI + 8;                             // gy columns of an image in LDS: 8 zeros in front
    static constexpr int RPG = wg_f32t_gpitch(NBI, NI), NRG = 9;
    static constexpr int CHX = wg_f32t_chx(K, NBI, NI), CHG = wg_f32t_chg(NBI, NI);
    static constexpr size_t lds_bytes = (size_t)CS * (CHX + CHG);
    static constexpr int NLX = (4 * XC * NQ + NT - 1) / NT, NLG = (4 * NI * TW * NQ + NT - 1) / NT;
    static_assert(XC % 8 == 0 && TW % 8 == 0 && lds_bytes <= 160 * 1024 && NLG == 1 && (size_t)K * K * CS * 4 <= lds_bytes, "sizes");
};

struct WgF32Geom {
    int B, H, W, C, OH, OW, PH, PW, BR, nbands, ncolt, nslices, U, units;
};

template <int K, int NBI, int NI>
__device__ __forceinline__ void dwconv_wgrad_f32_body(const float* __restrict__ x, const float* __restrict__ gy,
                                                      float* __restrict__ part, const WgF32Geom& g, int blk, int nblk) {
    using Sh = WgF32Shape<K, NBI, NI>;
    constexpr int NT = Sh::NT, CS = Sh::CS, NQ = Sh::NQ, NBV = Sh::NBV, COMB = Sh::COMB, NMF = Sh::NMF, XG = Sh::XG, TW = Sh::TW, XC = Sh::XC, XCI = Sh::XCI, GCI = Sh::GCI;
    constexpr int RPX = Sh::RPX, NRX = Sh::NRX, RPG = Sh::RPG, NRG = Sh::NRG, CHX = Sh::CHX, CHG = Sh::CHG, NLX = Sh::NLX;
    typedef float f4 __attribute__((ext_vector_type(4)));
    extern __shared__ uint32_t smem[];
    char* const xl = reinterpret_cast<char*>(smem);
    char* const gl = xl + CS * CHX;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int bid = xcd_remap(blk, nblk);
    const int sl = bid % g.nslices, chunk = bid / g.nslices, c0 = sl * CS;
    const int u0 = chunk * g.U, u1 = min(u0 + g.U, g.units);
    const long long img_x = (long long)g.H * g.W * g.C, img_g = (long long)g.OH * g.OW * g.C;
    constexpr uint32_t kNoRow = 0x80000000u;

    // ---- a thread's items: NLX of x, one of gy; (row of the group, image, column, channel quad)
    int xrow[NLX], xcol[NLX], xdst[NLX];
    uint32_t ximg[NLX];
    const int q = tid % NQ;
    const bool qok = c0 + 4 * q < g.C;
#pragma unroll
    for (int l = 0; l < NLX; ++l) {
        const int idx = (tid + l * NT) / NQ;
        const int c = idx % XC;
        xcol[l] = c % XCI, xrow[l] = idx / XC;
        ximg[l] = (uint32_t)(c / XCI) * (uint32_t)img_x + (uint32_t)(c0 + 4 * q);
        xdst[l] = 4 * q * CHX + (xrow[l] & 3) * RPX + c * 4;
    }
    const int gcol = (tid / NQ) % TW, gi_ = (tid / NQ) / TW % NI, grow = (tid / NQ) / TW / NI;
    const uint32_t gimg = (uint32_t)gi_ * (uint32_t)img_g + (uint32_t)(c0 + 4 * q);
    const int gdst = 4 * q * CHG + (gi_ * GCI + 8 + gcol) * 4;

    // the unit and group that is requested next
    struct Cursor {
        int u, ct, band, b, gi, ng, rows, orow0;
        __amdgpu_buffer_rsrc_t xr, gr;
    } cur;
    uint32_t xoff[NLX], goff;   // a thread's items in the unit: bytes from the group's first row, or kNoRow
    auto steps = [&](int band) { return (min(g.BR, g.OH - band * g.BR) + 4) / 4 + XG - 1; };   // over rows 0 .. rows, and the groups ahead of the first
    auto open = [&]() {
        const int ocol0 = cur.ct * TW, nimg = min(NI, g.B - cur.b);
        cur.orow0 = cur.band * g.BR;
        cur.rows = min(g.BR, g.OH - cur.orow0);
        cur.gi = 0, cur.ng = steps(cur.band);
        cur.xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x + cur.b * img_x), (short)0, (int)(nimg * img_x * 4), 0x00020000);
        cur.gr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(gy + cur.b * img_g), (short)0, (int)(nimg * img_g * 4), 0x00020000);
#pragma unroll
        for (int l = 0; l < NLX; ++l) {
            const int ic = ocol0 - g.PW + xcol[l];
            const bool ok = qok && xrow[l] < 4 && ic >= 0 && ic < g.W;
            xoff[l] = ok ? ((uint32_t)((xrow[l] * g.W + ic) * g.C) + ximg[l]) * 4u : kNoRow;
        }
        const bool ok = qok && grow < 4 && gcol < min(TW, g.OW - ocol0);
        goff = ok ? ((uint32_t)((grow * g.OW + ocol0 + gcol) * g.C) + gimg) * 4u : kNoRow;
    };
    f4 bx[2][NLX], bg[2];
    auto issue = [&](f4 (&dx)[NLX], f4& dg) {
        const int xr0 = cur.orow0 - g.PH + 4 * cur.gi, gr0 = 4 * (cur.gi - (XG - 1));
        const int xrow_at = xr0 * g.W * g.C * 4, grow_at = (cur.orow0 + gr0) * g.OW * g.C * 4;
        // where all four rows exist, nothing to compute per thread
        uint32_t xo[NLX], go = goff;
        int xs = xrow_at, gs = grow_at;
#pragma unroll
        for (int l = 0; l < NLX; ++l) xo[l] = xoff[l];
        if (xr0 < 0 || xr0 + 3 >= g.H) {   // (uniform, as the next)
            xs = 0;
#pragma unroll
            for (int l = 0; l < NLX; ++l) {
                const bool ok = (int)xoff[l] >= 0 && (unsigned)(xr0 + xrow[l]) < (unsigned)g.H;
                xo[l] = ok ? xoff[l] + (uint32_t)xrow_at : kNoRow;
            }
        }
        if (gr0 < 0 || gr0 + 3 >= cur.rows) {
            const bool ok = (int)goff >= 0 && (unsigned)(gr0 + grow) < (unsigned)cur.rows;
            gs = 0, go = ok ? goff + (uint32_t)grow_at : kNoRow;
        }
#pragma unroll
        for (int l = 0; l < NLX; ++l) dx[l] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(cur.xr, (int)xo[l], xs, 0));
        dg = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(cur.gr, (int)go, gs, 0));
        if (++cur.gi == cur.ng) {   // (uniform)
            if (++cur.u < u1) {
                if (++cur.ct == g.ncolt) {
                    cur.ct = 0;
                    if (++cur.band == g.nbands) cur.band = 0, cur.b += NI;
                }
                open();
            } else {   // past the last unit (at most four more requests): rows that no image has, which take no scalar offset
                cur.orow0 = g.PH - 64, cur.rows = 0, cur.gi = 0;
            }
        }
    };
    auto put = [&](char* d, int ch, const f4& v) {
        const float e0 = v.x, e1 = v.y, e2 = v.z, e3 = v.w;
        *reinterpret_cast<float*>(d) = e0, *reinterpret_cast<float*>(d + ch) = e1;
        *reinterpret_cast<float*>(d + 2 * ch) = e2, *reinterpret_cast<float*>(d + 3 * ch) = e3;
    };
    auto commit = [&](const f4 (&dx)[NLX], const f4& dg, int xslot, int grow0) {   // grow0: ring row of the group's first gy row
#pragma unroll
        for (int l = 0; l < NLX; ++l)
            if (wv * 64 + l * NT < 4 * XC * NQ) put(xl + xdst[l] + xslot * 4 * RPX, CHX, dx[l]);   // (whole wavefronts)
        int r = grow0 + (grow & 3);
        r -= r >= NRG ? NRG : 0;
        if (wv * 64 < 4 * NI * TW * NQ) put(gl + gdst + r * RPG, CHG, dg);
    };
    auto lds_barrier = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    cur.u = u0, cur.ct = u0 % g.ncolt, cur.band = u0 / g.ncolt % g.nbands, cur.b = u0 / g.ncolt / g.nbands * NI;
    int ct = cur.ct, band = cur.band;   // of the unit that is multiplied
    open();
    issue(bx[0], bg[0]);
    issue(bx[1], bg[1]);
    for (int i = tid; i < CS * CHG / 16; i += NT) reinterpret_cast<f4*>(gl)[i] = f4{0.f, 0.f, 0.f, 0.f};   // (gy's zero margins stay)
    lds_barrier();
    commit(bx[0], bg[0], 0, 0);
    issue(bx[0], bg[0]);

    // ---- operands of this wavefront's channel: lane = (m or n, k group kg)
    const int ln = lane & 15, kg = lane >> 4;
    uint32_t arow[NMF];   // bytes from the window's first row
    const char* abase[NMF];
#pragma unroll
    for (int f = 0; f < NMF; ++f) {
        const int mi = min(ln + 16 * f, COMB - 1);
        arow[f] = (uint32_t)(2 * (mi / NBV) * RPX);
        abase[f] = xl + wv * CHX + (8 * (mi % NBV) + 4 * kg) * 4;
    }
    const int du = ln >> 3, dv = ln & 7;
    const uint32_t bbase = (uint32_t)(CS * CHX + wv * CHG + (8 + 4 * kg - dv) * 4 - du * RPG);   // bytes in LDS
    const uint32_t bwrap = du ? NRG * RPG : 0;
    f4 acc[NMF][4], sum[NMF];   // of the last kFlush ticks; of all before
#pragma unroll
    for (int f = 0; f < NMF; ++f) {
        sum[f] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[f][t] = f4{0.f, 0.f, 0.f, 0.f};
    }
    auto flush = [&]() {
#pragma unroll
        for (int f = 0; f < NMF; ++f) {
            sum[f] += (acc[f][0] + acc[f][1]) + (acc[f][2] + acc[f][3]);
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[f][t] = f4{0.f, 0.f, 0.f, 0.f};
        }
    };
    // A block of 16 positions is a piece: the operands of the piece kAhead further on are read while one is multiplied.
    constexpr int NB = NBI * NI, kAhead = 1, kFlush = 4;
    struct Piece {
        f4 a[NMF];
        float b[4];
    };
    auto compute = [&](int xslot, int grow0) {   // where the tick's own groups (the newest) lie
        int xr0 = 4 * (xslot - (XG - 1));
        xr0 += xr0 < 0 ? NRX : 0;
        uint32_t bp = 0;
        const char* ap[NMF] = {};
        auto fetch = [&](Piece& o, int p) {
            const int ii = p / NB, nb = p % NB;
            if (nb == 0) {
                // gy row grow0 + ii - du of the ring: one further up where that is row -1
                const int gr = grow0 + ii - (grow0 + ii >= NRG ? NRG : 0);
                bp = bbase + (uint32_t)(gr * RPG) + (bwrap & (gr == 0 ? ~0u : 0u));
                asm("" : "+v"(bp));   // (whole in a register: with the planes' offset left to the reads, each adds it again)
                // window row xr0 + ii + 2a of the ring, whose rows come in pairs
#pragma unroll
                for (int f = 0; f < NMF; ++f) {
                    if (ii % 2 == 0) {
                        const uint32_t r = arow[f] + (uint32_t)((xr0 + ii) * RPX);
                        ap[f] = abase[f] + min(r, r - (uint32_t)(NRX * RPX));
                    } else {
                        ap[f] += RPX;
                    }
                }
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) o.b[t] = *reinterpret_cast<const float*>(xl + bp + 4 * (nb / NBI * GCI + nb % NBI * 16) + 4 * t);
#pragma unroll
            for (int f = 0; f < NMF; ++f) o.a[f] = *reinterpret_cast<const f4*>(ap[f] + 4 * (nb / NBI * XCI + nb % NBI * 16));
        };
        auto multiply = [&](const Piece& o) {
#pragma unroll
            for (int f = 0; f < NMF; ++f) {
                const float a0 = o.a[f].x, a1 = o.a[f].y, a2 = o.a[f].z, a3 = o.a[f].w;
                acc[f][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, o.b[0], acc[f][0], 0, 0, 0);
                acc[f][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, o.b[1], acc[f][1], 0, 0, 0);
                acc[f][2] = __builtin_amdgcn_mfma_f32_16x16x4f32(a2, o.b[2], acc[f][2], 0, 0, 0);
                acc[f][3] = __builtin_amdgcn_mfma_f32_16x16x4f32(a3, o.b[3], acc[f][3], 0, 0, 0);
            }
        };
        Piece pc[kAhead + 1];
#pragma unroll
        for (int p = 0; p < kAhead; ++p) fetch(pc[p], p);
#pragma unroll
        for (int p = 0; p < 4 * NB; ++p) {
            if (p + kAhead < 4 * NB) fetch(pc[(p + kAhead) % (kAhead + 1)], p + kAhead);
            __builtin_amdgcn_sched_barrier(0);
            multiply(pc[p % (kAhead + 1)]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // ---- ticks: group gi of a unit is in place; the products follow once XG groups of the unit are
    int xslot = 0, gslot = 0, gi = 0, u = u0, ng = steps(band);   // (gslot: ring row)
    auto tick = [&](f4 (&dx)[NLX], f4& dg) {   // (one past the last unit's: zeros into the rings)
        lds_barrier();
        if (gi % kFlush == 0) flush();   // (short chains of additions, however many units a workgroup takes)
        const int xn = xslot + 1 == XG + 1 ? 0 : xslot + 1, gn = gslot + 4 >= NRG ? gslot + 4 - NRG : gslot + 4;
        const bool mul = gi >= XG - 1 && u < u1;
        if (wv < CS / 2 && mul) compute(xslot, gslot);
        commit(dx, dg, xn, gn);
        issue(dx, dg);
        if (wv >= CS / 2 && mul) compute(xslot, gslot);
        xslot = xn, gslot = gn;
        if (++gi == ng) {
            if (++ct == g.ncolt) {
                ct = 0;
                if (++band == g.nbands) band = 0;
            }
            gi = 0, ng = steps(band), ++u;
        }
    };
    // (the two buffers by name and no way out between them: the compiler can then tell which requests are the newest, and a
    // commit waits for its own alone)
    do {
        tick(bx[1], bg[1]);
        tick(bx[0], bg[0]);
    } while (u < u1);
    flush();
    // ---- taps through LDS: [tap][channel], then 16-byte stores
    lds_barrier();
    float* const tl = reinterpret_cast<float*>(xl);
#pragma unroll
    for (int f = 0; f < NMF; ++f) {
        const float e[4] = {sum[f].x, sum[f].y, sum[f].z, sum[f].w};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int mi = 16 * f + 4 * kg + r, u = 2 * (mi / NBV) + du, v = 8 * (mi % NBV) + dv;
            if (mi < COMB && u < K && v < K) tl[(u * K + v) * CS + wv] = e[r];
        }
    }
    lds_barrier();
    for (int i = tid; i < K * K * NQ; i += NT) {
        if (c0 + 4 * (i % NQ) < g.C)
            *reinterpret_cast<f4*>(part + ((long long)chunk * K * K + i / NQ) * g.C + c0 + 4 * (i % NQ)) =
                *reinterpret_cast<const f4*>(tl + i / NQ * CS + 4 * (i % NQ));
    }
}

template <int K, int NBI, int NI>
constexpr int wg_f32t_waves() {
    return WgF32Shape<K, NBI, NI>::lds_bytes <= 80 * 1024 ? 4 : 2;
}

template <int K, int NBI, int NI>
__global__ __launch_bounds__(512, (wg_f32t_waves<K, NBI, NI>())) void dwconv_wgrad_f32t_k(const float* __restrict__ x, const float* __restrict__ gy,
                                                                                    float* __restrict__ part, const WgF32Geom g) {
    dwconv_wgrad_f32_body<K, NBI, NI>(x, gy, part, g, blockIdx.x, gridDim.x);
}

// ------------------------------------------------------------------------------------------------
// Host side

struct WgF32Plan {
    WgF32Geom g;
    int nbi;             // 16-column blocks of a tile (4, 3, or 2 and 1 with two and four images side by side)
    int nchunks;         // partials
    bool ok;
};

// The plan depends on the shape alone (the workspace is sized by it).
inline WgF32Plan wgrad_f32t_plan(int B, int H, int W, int C, int K, int PH, int PW) {
    WgF32Plan p{};
    p.g = WgF32Geom{B, H, W, C, H + 2 * PH - K + 1, W + 2 * PW - K + 1, PH, PW, 0, 1, 0, 0, 1, 0};
    WgF32Geom& g = p.g;
    // Where the vector-ALU kernel (dwconv_wgrad_tiled.h) stays faster: images narrower than a 16-position block is worth
    // ([38,9,9,184] filter 9: 28 us here, 20 there; filter 17 50 and 51), and filters up to 9 on large tensors, where it
    // takes time by the tap and this kernel by the position ([32,56,56,64] filter 7: 55 here, 39 there; filter 11 on: 55
    // here, 60 .. 80 there; [32,28,28,64] filter 7: 26 here, 36 there).
    if (K < 15 && (g.OW < 12 || (K < 11 && (long long)B * g.OH * g.OW * C > 3000000))) return p;
    if (B < 1 || g.OH < 1 || g.OW < 1 || C % 4 != 0 || K < 3 || K > 17 || !(K & 1)) return p;
    long long least = -1;
    for (int nbi = 4; nbi >= 1; --nbi) {   // tiles of 56, 40, 24 or 8 columns: the fewest blocks over the rows of all images
        const int ni = nbi > 2 ? 1 : 4 / nbi;
        const long long blocks = (long long)cdiv(g.OW, 16 * nbi - 8) * nbi * cdiv(B, ni) * ni;
        if (least < 0 || blocks < least) least = blocks, p.nbi = nbi;
    }
    const int ni = p.nbi > 2 ? 1 : 4 / p.nbi;
    if ((long long)H * W * C * ni > 0x1fffffffLL || (long long)g.OH * g.OW * C * ni > 0x1fffffffLL) return p;
    g.ncolt = cdiv(g.OW, 16 * p.nbi - 8), g.nslices = cdiv(C, 8);
    // One, two or three workgroups for every compute unit: bands of an image, or several units each; the cheapest by the
    // cycles of a unit's ticks (with products: 4 rows of the tile by two wavefronts and what the other workgroup's products do
    // not cover of the staging; without: 800) and of the start-up (9000, half for each further round), the fewer workgroups
    // where they tie.  As one of a pair, which is how a block runs it, a problem leaves the compute units that it does not fill
    // to the other, so that half of its price is its work and half its longest unit (us of the pair, two workgroups each -> by
    // this rule: [32,56,56,64] filter 13 62.9 -> 55.6, [16,28,28,96] filter 9 29.8 -> 27.0, [64,40,40,32] filter 9 75 -> 63).
    // The same plan by itself and in a pair: the results are then the same to the bit.
    const int units = cdiv(B, ni) * g.ncolt, nmf = ((K + 1) / 2 * ((K + 7) / 8) + 15) / 16, xg = (4 + 2 * ((K + 1) / 2 - 1) + 3) / 4;
    const int held = 8 * (wg_f32t_chx(K, p.nbi, ni) + wg_f32t_chg(p.nbi, ni)) <= 80 * 1024 ? 2 : 1;
    double least_cost = -1;
    for (int n = 1; n <= 3; ++n) {
        int c = 256 * n / g.nslices, br = g.OH, u = 1;   // chunks of a slice
        if (c < 1) c = 1;
        if (c > units) {
            int nb = c / units;
            if (nb > cdiv(g.OH, 4)) nb = cdiv(g.OH, 4);
            if (nb > 1) br = (cdiv(g.OH, nb) + 1 + 3) / 4 * 4 - 1;   // (rows + 1 whole groups of four)
        } else {
            u = cdiv(units, c);
        }
        const int nbands = cdiv(g.OH, br), chunks = cdiv(units * nbands, u);
        const long long each = cdiv((long long)chunks * g.nslices, 256);   // workgroups of a compute unit
        const double fill = (double)((long long)chunks * g.nslices) / 256;
        const double cost = 0.5 * (each + (fill > 0.8 ? fill : 0.8)) * u * (((br + 4) / 4) * (1024 * p.nbi * ni * nmf + 400) + (xg - 1) * 800) +
                            4500.0 * (1 + cdiv(each, held));
        if (least_cost < 0 || cost < 0.98 * least_cost) least_cost = cost, g.BR = br, g.U = u;
    }
    if (const char* e = tune_env("PDW_WGF")) sscanf(e, "%d,%d", &g.BR, &g.U);
    g.nbands = cdiv(g.OH, g.BR);
    g.units = units * g.nbands;
    p.nchunks = cdiv(g.units, g.U);
    p.ok = (long long)p.nchunks * g.nslices <= 0x7fffffffLL;
    return p;
}

// -1: not covered.  ws: nchunks * K * K * C floats.
template <int K>
int launch_wgrad_f32t(const void* x, const void* gy, void* dw, void* ws, int B, int H, int W, int C, int PH, int PW, hipStream_t s) {
    const WgF32Plan p = wgrad_f32t_plan(B, H, W, C, K, PH, PW);
    if (!p.ok) return -1;
    for (const void* q : {x, gy, (const void*)ws})
        if (reinterpret_cast<uintptr_t>(q) & 15) return -1;
    const dim3 grid((unsigned)(p.nchunks * p.g.nslices));
#define PDW_WGF32(NBI, NI)                                                                                                 \
    {                                                                                                                      \
        auto kern = dwconv_wgrad_f32t_k<K, NBI, NI>;                                                                       \
        static std::once_flag once;                                                                                        \
        std::call_once(once, [&] { (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); }); \
        constexpr size_t lds = WgF32Shape<K, NBI, NI>::lds_bytes;                                                          \
        hipLaunchKernelGGL(kern, grid, dim3(512), lds, s, (const float*)x, (const float*)gy, (float*)ws, p.g);             \
    }
    switch (p.nbi) {
        case 4: PDW_WGF32(4, 1) break;
        case 3: PDW_WGF32(3, 1) break;
        case 2: PDW_WGF32(2, 2) break;
        default: PDW_WGF32(1, 4)
    }
#undef PDW_WGF32
    if (int e = check_launch("dwconv_wgrad_f32t")) return e;
    return wgrad_reduce_launch<float>((const float*)ws, (float*)dw, p.nchunks, K * K * C, s);
}

// The weight gradients of two problems (a block's scales) in one grid, each in the tile of its plan: neither depends on the
// other, and where one of them leaves compute units without work the launch takes as long as the longer one (us with the
// summations, at the start of both and now: [2,32,32,32] and its half scale, filter 7, 16.1 -> 13.8; [3,57,61,100], filter 15,
// 29.9 -> 23.6; [32,56,56,64], filter 13, 77 -> 55.6; [4,64,64,576], filter 13, 126.5 -> 106.7).
struct WgF32Problem {
    const float *x, *gy;
    float* part;
    WgF32Geom g;
    int nbi, n;   // 16-column blocks of a tile; workgroups
};
struct WgF32Pair {
    WgF32Problem p[2];
    MeanJob mean;   // workgroups behind both problems: the backward of the block's mean branch, which needs nothing of this
};                  // launch and whose result is read after it (by a launch of its own 5.1 us at [32,56,56,128], 3.1 at [2,32,32,64])

// Tiles that leave room for two workgroups on a compute unit: the pair is for those.
template <int K>
constexpr bool wg_f32t_pairs(int nbi) {
    return (nbi == 4   ? wg_f32t_waves<K, 4, 1>()
            : nbi == 3 ? wg_f32t_waves<K, 3, 1>()
            : nbi == 2 ? wg_f32t_waves<K, 2, 2>()
                       : wg_f32t_waves<K, 1, 4>()) == 4;
}

template <int K>
__device__ __forceinline__ void wgrad_f32t_pair_body(const WgF32Pair& a, int blk) {
    const bool first = blk < a.p[0].n;
    const float *x = first ? a.p[0].x : a.p[1].x, *gy = first ? a.p[0].gy : a.p[1].gy;
    float* const part = first ? a.p[0].part : a.p[1].part;
    const WgF32Geom g = first ? a.p[0].g : a.p[1].g;
    const int nbi = first ? a.p[0].nbi : a.p[1].nbi, at = blk - (first ? 0 : a.p[0].n), n = first ? a.p[0].n : a.p[1].n;
    if constexpr (wg_f32t_pairs<K>(4))
        if (nbi == 4) return dwconv_wgrad_f32_body<K, 4, 1>(x, gy, part, g, at, n);
    if constexpr (wg_f32t_pairs<K>(3))
        if (nbi == 3) return dwconv_wgrad_f32_body<K, 3, 1>(x, gy, part, g, at, n);
    if constexpr (wg_f32t_pairs<K>(2))
        if (nbi == 2) return dwconv_wgrad_f32_body<K, 2, 2>(x, gy, part, g, at, n);
    if constexpr (wg_f32t_pairs<K>(1))
        if (nbi == 1) return dwconv_wgrad_f32_body<K, 1, 4>(x, gy, part, g, at, n);
}

template <int K>
__global__ __launch_bounds__(512, 4) void dwconv_wgrad_f32t_pair_k(const WgF32Pair a) {
    if ((int)blockIdx.x >= a.p[0].n + a.p[1].n) {
        extern __shared__ uint32_t smem[];
        return mean_bwd_body<float, 512, false>(a.mean, (int)blockIdx.x - a.p[0].n - a.p[1].n, reinterpret_cast<float*>(smem));
    }
    wgrad_f32t_pair_body<K>(a, blockIdx.x);
}

// And with the input gradient of the second problem (dwconv_f32t.h), which the launch behind this one adds: by itself one workgroup a compute
// unit with half of its time in start-up and last steps.  It lies where the weight gradients' workgroups end and fills the places of their
// last round, or in front (d0 = 0) where that is (nearly) full, since it would be a round of its own then: as its shorter workgroups
// end, places come free one after the other.  us, the input gradient + the weight gradients -> this: [2,32,32,32] filter 7 (its half scale's)
// 5.8 + 9.7 -> 9.6; [2,92,92,104] filter 11 9.5 + 24.2 -> 26.4 (in front 29.9); [64,28,28,48] filter 13 10.3 + 45.7 -> 46.8 (50.4);
// [32,56,56,64] filter 13 15.7 + 56.4 -> 66.5 (behind 74.7); [16,56,56,64] 37.3 (43.4), filter 15 11.7 + 32.9 -> 40.3.
template <int K>
__global__ __launch_bounds__(512, 4) void dwconv_bwd_f32t_half_k(const WgF32Pair a, const F32Problem d, int d0) {
    const int blk = (int)blockIdx.x, at = blk - d0, nw = a.p[0].n + a.p[1].n;
    if (blk >= nw + d.n) {
        extern __shared__ uint32_t smem[];
        return mean_bwd_body<float, 512, false>(a.mean, blk - nw - d.n, reinterpret_cast<float*>(smem));
    }
    if (at < 0 || at >= d.n) return wgrad_f32t_pair_body<K>(a, at < 0 ? blk : blk - d.n);
    if (d.npc == 16) dwconv_f32_body<K, 16, 0>(d.x, d.w, nullptr, d.y, d.g, at, d.n);
    else if (d.npc == 8) dwconv_f32_body<K, 8, 0>(d.x, d.w, nullptr, d.y, d.g, at, d.n);
    else dwconv_f32_body<K, 4, 0>(d.x, d.w, nullptr, d.y, d.g, at, d.n);
}

// -1: not covered (the caller makes two launches).  w1, dx1 (optional): the second problem's filter and input gradient.
template <int K>
int launch_wgrad_f32t_pair(const void* x0, const void* gy0, void* dw0, void* ws0, int H0, int W0, const void* x1, const void* gy1,
                           void* dw1, void* ws1, int H1, int W1, int B, int C, int P, hipStream_t s, const MeanJob* mean, const void* w1, void* dx1) {
    const WgF32Plan plan[2] = {wgrad_f32t_plan(B, H0, W0, C, K, P, P), wgrad_f32t_plan(B, H1, W1, C, K, P, P)};
    const void *const x[2] = {x0, x1}, *const gy[2] = {gy0, gy1};
    void *const dw[2] = {dw0, dw1}, *const ws[2] = {ws0, ws1};
    WgF32Pair a{};
    size_t lds = 0;
    long long n = 0;
    for (int i = 0; i < 2; ++i) {
        const WgF32Plan& p = plan[i];
        if (!p.ok || !wg_f32t_pairs<K>(p.nbi)) return -1;
        for (const void* q : {x[i], gy[i], (const void*)ws[i]})
            if (reinterpret_cast<uintptr_t>(q) & 15) return -1;
        const int mine = p.nchunks * p.g.nslices;
        a.p[i] = WgF32Problem{(const float*)x[i], (const float*)gy[i], (float*)ws[i], p.g, p.nbi, mine};
        n += mine;
        const size_t need = p.nbi == 4   ? WgF32Shape<K, 4, 1>::lds_bytes
                            : p.nbi == 3 ? WgF32Shape<K, 3, 1>::lds_bytes
                            : p.nbi == 2 ? WgF32Shape<K, 2, 2>::lds_bytes
                                         : WgF32Shape<K, 1, 4>::lds_bytes;
        if (need > lds) lds = need;
    }
    if (mean) {
        const size_t need = mean_lds(mean->D, 512);
        if (need > 80 * 1024) return -1;   // (two workgroups on a compute unit)
        if (need > lds) lds = need;
        a.mean = *mean, n += (long long)mean->B * mean_slices(mean->D);
    }
    F32Problem d{};
    if (dx1) {
        long long nd;
        if (!f32t_problem<K>(d, nd, lds, gy1, w1, dx1, B, H1, W1, C, true)) return -1;
        n += nd;
    }
    const long long nw = a.p[0].n + a.p[1].n;
    const int d0 = (nw + 511) % 512 + 1 >= 448 ? 0 : (int)nw;   // (two workgroups a compute unit: 512 a round)
    if (n > 0x7fffffffLL) return -1;
    static std::once_flag once;
    std::call_once(once, [] {
        (void)hipFuncSetAttribute((const void*)dwconv_wgrad_f32t_pair_k<K>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)hipFuncSetAttribute((const void*)dwconv_bwd_f32t_half_k<K>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    });
    if (!dx1) hipLaunchKernelGGL(dwconv_wgrad_f32t_pair_k<K>, dim3((unsigned)n), dim3(512), lds, s, a);
    else hipLaunchKernelGGL(dwconv_bwd_f32t_half_k<K>, dim3((unsigned)n), dim3(512), lds, s, a, d, d0);
    if (int e = check_launch("dwconv_wgrad_f32t_pair")) return e;
    for (int i = 0; i < 2; ++i)
        if (int e = wgrad_reduce_launch<float>((const float*)ws[i], (float*)dw[i], plan[i].nchunks, K * K * C, s)) return e;
    return 0;
}

}  // namespace pdw
