// Depthwise weight gradient in fp32 on the fp32 matrix cores: stride 1, dilation 1, odd square filters 3 .. 17.
//
// As in dwconv_wgrad_tz.h, with u = 2a + du, v = 8b + dv:  dw[2a+du][8b+dv] = sum over p of xw[p + (2a,8b)] gy[p - (du,dv)],
// one v_mfma_f32_16x16x4_f32 with m = (a,b), n = (du,dv), k = 4 positions: an accumulator of 4 registers holds all taps of a
// channel (filter 17: 27 (a,b), two instructions that share the gy operand).  Four instructions take 16 positions of a row:
// position 4g + t of the block for lane group g in instruction t, so that a lane's four xw values are one aligned
// 16-byte LDS read, and its four gy values two 8-byte pairs at any element offset.
//
// What bounds it: the matrix pipe (32 cycles an instruction; its operands cost the LDS half of that).  Every position of a
// row block costs the same whatever the filter, and a row block computes 16 positions of which 8 per tile are margin.
//
// A workgroup (8 wavefronts, one channel each) takes `U` units (image, row band, column tile) of one 8-channel slice one
// after the other as one stream: a tick brings four window rows of x and four rows of gy into LDS rings (requested two
// ticks ahead, across units as well) while the previous ones are multiplied, so only the first unit of a workgroup waits
// for memory.  The taps leave through LDS as 16-byte stores into the workgroup's partial; fixed-order summation, no atomics.
//
// Measured with the summation at [32,56,56,64]: filter 13 55 us for 78 on the vector ALU (dwconv_wgrad_tiled.h), 17 95 for
// 177; [32,28,28,64]: filter 3 24 for 43, 13 27 for 33.  The products alone are 29 and the staging alone 29 of the 51 us
// (filter 13, without the summation): the matrix pipe is 57 % busy.  16 channels a workgroup for whole 64-byte requests
// measured the same.
#pragma once
#include <mutex>

#include "common.h"
#include "kernels.h"
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
    static_assert(lds_bytes <= 160 * 1024 && NLG == 1 && (size_t)K * K * CS * 4 <= lds_bytes, "sizes");
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
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
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
        int u, gi, ng, rows, orow0, ocol0, cols;
        __amdgpu_buffer_rsrc_t xr, gr;
    } cur;
    auto open = [&](int u) {
        cur.u = u, cur.gi = 0;
        const int ct = u % g.ncolt, t = u / g.ncolt, band = t % g.nbands, b = t / g.nbands * NI;
        const int nimg = u < u1 ? min(NI, g.B - b) : 0;
        cur.orow0 = band * g.BR, cur.ocol0 = ct * TW;
        cur.rows = min(g.BR, g.OH - cur.orow0), cur.cols = min(TW, g.OW - cur.ocol0);
        cur.ng = (cur.rows + 4) / 4 + XG - 1;   // steps over rows 0 .. rows, and the groups ahead of the first
        cur.xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x + (nimg ? b : 0) * img_x), (short)0, (int)(nimg * img_x * 4), 0x00020000);
        cur.gr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(gy + (nimg ? b : 0) * img_g), (short)0, (int)(nimg * img_g * 4), 0x00020000);
    };
    f4 bx[2][NLX], bg[2];
    auto issue = [&](f4 (&dx)[NLX], f4& dg) {
#pragma unroll
        for (int l = 0; l < NLX; ++l) {
            const int ic = cur.ocol0 - g.PW + xcol[l], ir = cur.orow0 - g.PH + 4 * cur.gi + xrow[l];
            const bool ok = qok && xrow[l] < 4 && ic >= 0 && ic < g.W && ir >= 0 && ir < g.H;
            const uint32_t off = ok ? ((uint32_t)((ir * g.W + ic) * g.C) + ximg[l]) * 4u : kNoRow;
            dx[l] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(cur.xr, (int)off, 0, 0));
        }
        const int r = 4 * (cur.gi - (XG - 1)) + grow;
        const bool ok = qok && grow < 4 && gcol < cur.cols && r >= 0 && r < cur.rows;
        const uint32_t off = ok ? ((uint32_t)(((cur.orow0 + r) * g.OW + cur.ocol0 + gcol) * g.C) + gimg) * 4u : kNoRow;
        dg = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(cur.gr, (int)off, 0, 0));
        if (++cur.gi == cur.ng) open(cur.u + 1);   // (uniform; past the last unit: empty descriptors)
    };
    auto put = [&](char* d, int ch, const f4& v) {
        const float e0 = v.x, e1 = v.y, e2 = v.z, e3 = v.w;
        *reinterpret_cast<float*>(d) = e0, *reinterpret_cast<float*>(d + ch) = e1;
        *reinterpret_cast<float*>(d + 2 * ch) = e2, *reinterpret_cast<float*>(d + 3 * ch) = e3;
    };
    auto commit = [&](const f4 (&dx)[NLX], const f4& dg, int xslot, int grow0) {   // grow0: ring row of the group's first gy row
#pragma unroll
        for (int l = 0; l < NLX; ++l)
            if (xrow[l] < 4) put(xl + xdst[l] + xslot * 4 * RPX, CHX, dx[l]);
        int r = grow0 + (grow & 3);
        r -= r >= NRG ? NRG : 0;
        if (grow < 4) put(gl + gdst + r * RPG, CHG, dg);
    };
    auto lds_barrier = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    open(u0);
    issue(bx[0], bg[0]);
    issue(bx[1], bg[1]);
    // the zero margins of gy: everything but the tiles' own columns
    for (int i = tid; i < CS * NRG * (RPG / 4); i += NT) {
        const int c = i % (RPG / 4), row = i / (RPG / 4) % NRG, ch = i / (RPG / 4) / NRG;
        if (c >= NI * GCI || c % GCI < 8 || c % GCI >= 8 + TW) *reinterpret_cast<float*>(gl + ch * CHG + row * RPG + c * 4) = 0.f;
    }
    commit(bx[0], bg[0], 0, 0);
    issue(bx[0], bg[0]);

    // ---- operands of this wavefront's channel: lane = (m or n, k group kg)
    const int ln = lane & 15, kg = lane >> 4;
    int arow[NMF];
    const char* abase[NMF];
#pragma unroll
    for (int f = 0; f < NMF; ++f) {
        const int mi = min(ln + 16 * f, COMB - 1);
        arow[f] = 2 * (mi / NBV);
        abase[f] = xl + wv * CHX + (8 * (mi % NBV) + 4 * kg) * 4;
    }
    const int du = ln >> 3, dv = ln & 7;
    const char* const bbase = gl + wv * CHG + (8 + 4 * kg - dv) * 4;
    f4 acc[NMF][4];
#pragma unroll
    for (int f = 0; f < NMF; ++f)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[f][t] = f4{0.f, 0.f, 0.f, 0.f};
    // With one product a position, a row's operands are read while the previous row is multiplied (left to itself the
    // compiler reads a block's operands, waits for them and multiplies); with two (K = 17) the operands of a row would not
    // fit the registers, and the second product covers the reads.
    struct Row {
        f4 a[NBI * NI][NMF];
        float b[NBI * NI][4];
    };
    auto compute = [&](int xslot, int grow0) {   // where the tick's own groups (the newest) lie
        int xr0 = 4 * (xslot - (XG - 1));
        xr0 += xr0 < 0 ? NRX : 0;
        auto fetch = [&](Row& o, int ii) {
            int gr = grow0 + ii - du;
            gr += gr < 0 ? NRG : 0;
            gr -= gr >= NRG ? NRG : 0;
            const char* bp = bbase + gr * RPG;
#pragma unroll
            for (int nb = 0; nb < NBI * NI; ++nb)
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    o.b[nb][t] = *reinterpret_cast<const float*>(bp + 4 * (nb / NBI * GCI + nb % NBI * 16) + 4 * t);
#pragma unroll
            for (int f = 0; f < NMF; ++f) {
                int r = xr0 + ii + arow[f];
                r -= r >= NRX ? NRX : 0;
                const char* ap = abase[f] + r * RPX;
#pragma unroll
                for (int nb = 0; nb < NBI * NI; ++nb) o.a[nb][f] = *reinterpret_cast<const f4*>(ap + 4 * (nb / NBI * XCI + nb % NBI * 16));
            }
        };
        auto multiply = [&](const Row& o) {
#pragma unroll
            for (int nb = 0; nb < NBI * NI; ++nb)
#pragma unroll
                for (int f = 0; f < NMF; ++f) {
                    const float a0 = o.a[nb][f].x, a1 = o.a[nb][f].y, a2 = o.a[nb][f].z, a3 = o.a[nb][f].w;
                    acc[f][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, o.b[nb][0], acc[f][0], 0, 0, 0);
                    acc[f][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, o.b[nb][1], acc[f][1], 0, 0, 0);
                    acc[f][2] = __builtin_amdgcn_mfma_f32_16x16x4f32(a2, o.b[nb][2], acc[f][2], 0, 0, 0);
                    acc[f][3] = __builtin_amdgcn_mfma_f32_16x16x4f32(a3, o.b[nb][3], acc[f][3], 0, 0, 0);
                }
        };
        Row row[NMF == 1 ? 2 : 1];
        if constexpr (NMF == 1) {
            fetch(row[0], 0);
#pragma unroll
            for (int ii = 0; ii < 4; ++ii) {
                if (ii < 3) fetch(row[(ii + 1) & 1], ii + 1);
                __builtin_amdgcn_sched_barrier(0);
                multiply(row[ii & 1]);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
#pragma unroll
            for (int ii = 0; ii < 4; ++ii) {
                fetch(row[0], ii);
                multiply(row[0]);
            }
        }
    };
    // ---- ticks: group gi of unit u is in place; the products follow once XG groups of the unit are
    int xslot = 0, gslot = 0, par = 1;   // (gslot: ring row)
    for (int u = u0; u < u1; ++u) {
        const int band = u / g.ncolt % g.nbands;
        const int ng = (min(g.BR, g.OH - band * g.BR) + 4) / 4 + XG - 1;
        for (int gi = 0; gi < ng; ++gi) {
            lds_barrier();
            const int xn = xslot + 1 == XG + 1 ? 0 : xslot + 1, gn = gslot + 4 >= NRG ? gslot + 4 - NRG : gslot + 4;
            const bool mul = gi >= XG - 1;
            if (wv < CS / 2 && mul) compute(xslot, gslot);
            if (par) {   // (uniform)
                commit(bx[1], bg[1], xn, gn);
                issue(bx[1], bg[1]);
            } else {
                commit(bx[0], bg[0], xn, gn);
                issue(bx[0], bg[0]);
            }
            if (wv >= CS / 2 && mul) compute(xslot, gslot);
            xslot = xn, gslot = gn, par ^= 1;
        }
    }
    // ---- taps through LDS: [tap][channel], then 16-byte stores
    lds_barrier();
    float* const tl = reinterpret_cast<float*>(xl);
#pragma unroll
    for (int f = 0; f < NMF; ++f) {
        const f4 s = (acc[f][0] + acc[f][1]) + (acc[f][2] + acc[f][3]);
        const float e[4] = {s.x, s.y, s.z, s.w};
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
    // two workgroups for every compute unit: several units each, or row bands of at least 12 rows (5 where those would not
    // give every compute unit one: the chain of a band's steps is all there is to wait for)
    const int want = 512;
    const long long whole = (long long)cdiv(B, ni) * g.ncolt * g.nslices;
    g.BR = g.OH;
    if (whole >= 2 * want) {
        g.U = (int)(whole / want);
    } else if (whole < want) {
        int nb = (int)(want / whole);
        const int least_rows = whole * (g.OH / 12) >= 256 ? 12 : 5;
        if (nb > g.OH / least_rows) nb = g.OH / least_rows;
        if (nb > 1) g.BR = (cdiv(g.OH, nb) + 1 + 3) / 4 * 4 - 1;   // (rows + 1 whole groups of four)
    }
    g.nbands = cdiv(g.OH, g.BR);
    g.units = cdiv(B, ni) * g.ncolt * g.nbands;
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
// other, and at the sizes where one of them leaves compute units without work the launch takes as long as the longer one
// ([2,32,32,32] and its half scale, filter 7, us: 10.6 + 12.4 -> 12.6; [3,57,61,100], filter 15: 25.2 + 12.0 -> 26.0;
// [32,56,56,64], filter 13, where both fill the chip: 57.5 + 25.6 -> 76.1).
struct WgF32Problem {
    const float *x, *gy;
    float* part;
    WgF32Geom g;
    int nbi, n;   // 16-column blocks of a tile; workgroups
};
struct WgF32Pair {
    WgF32Problem p[2];
};

// Tiles that leave room for two workgroups on a compute unit: the pair is for those.
template <int K>
constexpr bool wg_f32t_pairs(int nbi) {
    return (nbi == 4   ? wg_f32t_waves<K, 4, 1>()
            : nbi == 3 ? wg_f32t_waves<K, 3, 1>()
            : nbi == 2 ? wg_f32t_waves<K, 2, 2>()
                       : wg_f32t_waves<K, 1, 4>()) == 4;
}

template <int K>
__global__ __launch_bounds__(512, 4) void dwconv_wgrad_f32t_pair_k(const WgF32Pair a) {
    const bool first = (int)blockIdx.x < a.p[0].n;
    const float *x = first ? a.p[0].x : a.p[1].x, *gy = first ? a.p[0].gy : a.p[1].gy;
    float* const part = first ? a.p[0].part : a.p[1].part;
    const WgF32Geom g = first ? a.p[0].g : a.p[1].g;
    const int nbi = first ? a.p[0].nbi : a.p[1].nbi, at = (int)blockIdx.x - (first ? 0 : a.p[0].n), n = first ? a.p[0].n : a.p[1].n;
    if constexpr (wg_f32t_pairs<K>(4))
        if (nbi == 4) return dwconv_wgrad_f32_body<K, 4, 1>(x, gy, part, g, at, n);
    if constexpr (wg_f32t_pairs<K>(3))
        if (nbi == 3) return dwconv_wgrad_f32_body<K, 3, 1>(x, gy, part, g, at, n);
    if constexpr (wg_f32t_pairs<K>(2))
        if (nbi == 2) return dwconv_wgrad_f32_body<K, 2, 2>(x, gy, part, g, at, n);
    if constexpr (wg_f32t_pairs<K>(1))
        if (nbi == 1) return dwconv_wgrad_f32_body<K, 1, 4>(x, gy, part, g, at, n);
}

// -1: not covered (the caller makes two launches).
template <int K>
int launch_wgrad_f32t_pair(const void* x0, const void* gy0, void* dw0, void* ws0, int H0, int W0, const void* x1, const void* gy1,
                           void* dw1, void* ws1, int H1, int W1, int B, int C, int P, hipStream_t s) {
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
    if (n > 0x7fffffffLL) return -1;
    static std::once_flag once;
    std::call_once(once, [] {
        (void)hipFuncSetAttribute((const void*)dwconv_wgrad_f32t_pair_k<K>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    });
    hipLaunchKernelGGL(dwconv_wgrad_f32t_pair_k<K>, dim3((unsigned)n), dim3(512), lds, s, a);
    if (int e = check_launch("dwconv_wgrad_f32t_pair")) return e;
    for (int i = 0; i < 2; ++i)
        if (int e = wgrad_reduce_launch<float>((const float*)ws[i], (float*)dw[i], plan[i].nchunks, K * K * C, s)) return e;
    return 0;
}

}  // namespace pdw
