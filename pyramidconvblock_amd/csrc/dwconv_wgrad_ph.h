// Depthwise-convolution weight gradient on the dense matrix cores, phase-major (16-bit types, stride 1, dilation 1, square
// filters up to 17):     dw[u,v,c] = sum_{b,i,j} gy[b,i,j,c] * xw[b, i+u, j+v, c],   xw[r][s] = x[r-PH][s-PW].
//
// A row of 64 gy columns j = 8q + r is kept as 8 vectors G_r, r = j mod 8, of the 8 values q = 0..7, and a row of x as the
// vectors X_p[q] = xw[8q + p], p = 0 .. 7 + K-1.  A column offset of v is then another vector instead of a shift inside one,
//     dw[u][v] = sum over rows rho of x and phases r of  X_{r+v}[rho] . G_r[rho - u],
// and both operands of v_mfma_f32_16x16x32_{bf16,f16} (lane = index + 16 * k group, a k group = 8 values) are aligned 16-byte
// vectors: A holds X_{r+v} (index v, k group = one of 4 phases), B holds G_r of 16 rows (index = row mod 16).  One
// accumulator of 4 registers holds all taps of a channel, a row takes 2 products (8 phases) per channel.
//
// What bounds it: the LDS before anything else.  By the counters ([128,56,56,64] filter 13, 16 passes a run) it is busy 51 % of the
// cycles, a quarter of that bank conflicts, the vector ALU 26 % and the matrix pipe 21 %; wavefronts wait for their turn at the
// LDS a fifth of their time and for data or a barrier a third.  B stays in registers: from one row of x to the next only the
// gy row that enters changes (GR rows at a time, one read and four selects), so that a product costs one 16-byte LDS read per
// lane (4 cycles) instead of the 11 cycles of an aligned operand and one at single-element offsets.  The index of a gy row in B is fixed while
// u = rho - row moves with rho: there are 8 accumulators, by rho mod 8, whose lanes are rotated against each other when they are
// added at the end (DPP row rotates), and B itself is rotated by 8 lanes once in 8 rows.
//
// Rows are streamed through LDS in passes of 8 (double-buffered, requested two passes ahead).  The images of a batch are
// stacked into one column of rows, `per` rows apart with at least PH rows of zeros between them, and a workgroup takes a
// run of passes wherever it starts: as many workgroups as the chip holds at once, whatever the extents, one start-up each.
// Tiles of 64 columns of an image, or of 32 columns of two images side by side (the halves of the vectors).
// Fixed-order summation of the workgroups' partials (wgrad_reduce_parts), no atomics.
//
// us of the kernel (the summation is 4 more), against tiles of one image, gy shifted by elements: [8,64,64,1152] filter 9 139 -> 47 (its tiles are
// 56 columns wide, 1152 workgroups of one start-up each; 151 MB at 3.2 TB/s now), [32,56,56,64] filter 13 17.6 -> 15.4,
// [128,56,56,64] 50 -> 37, [128,7,7,1152] filter 3 166 -> 34.  With all of the chip in such runs a pass takes 1.8 us and a run 8 besides
// (4, 16 and 23 passes of 64 columns in the first three).
//
// Filters 16 and 17 have one more column and row than the indices.  The 16 rows of B are then those before x's row (u = 1 .. 16), and
// the rest comes from 8 products a pass besides the 32 of a channel: column 16 with the pass's 8 rows of x as A's index, row 0 with
// the vectors p against the phases r and the rows as k groups (both as differences of their indices, added up at the end by lane
// rotations: 10.1 us of the smallest launch, 10.9 through LDS).  us of kernel and summation against a kernel of two accumulators over bands
// of single images (two 1 KB operands a product): [32,56,56,64] 26.6 -> 19.9, [128,56,56,64] 77.4 -> 45.7, [5,47,51,1000] 64.3 -> 31.9,
// [79,7,7,264] 53.7 -> 21.1, [1,28,28,64] 10.0 -> 9.5.
#pragma once
#include <mutex>

#include "common.h"
#include "dwconv_tz.h"
#include "kernels.h"
#include "tile_common.h"

namespace pdw {

// NCOPY: 8-vector groups of an x row (p < 8 NCOPY: 2 up to K = 9, 3 beyond); GR: gy rows that enter B at a time
// (K + GR - 1 <= 16: a row that is in B too early multiplies into taps beyond the filter).  8: filters 16 and 17, the pass's rows are
// read at once and enter one by one, each after its own row of x.
template <int NCOPY, int GR>
struct WgPhShape {
    static constexpr int NT = 512, CS = 16, CPW = 2;
    static constexpr int XROW = 128 * NCOPY, XPL = 8 * XROW;   // bytes of an x row, of a channel's pass
    // gy rows 36 banks apart: the 4 rows x 4 phases a B read takes lie in different banks
    static constexpr int GROW = 144, GPL = 8 * GROW;
    static constexpr int HALF = 128;   // channels 8..15 sit 32 banks further: a staging write's two 8-channel pieces differ
    static constexpr int XBUF = CS * XPL + HALF, GBUF = CS * GPL + HALF;
    static constexpr size_t lds_bytes = 2 * (size_t)(XBUF + GBUF);
    static_assert((NCOPY == 2 || NCOPY == 3) && (GR == 2 || GR == 4 || GR == 8), "vector groups, rows per update");
    static_assert(XPL % 256 == 0 && GPL % 128 == 0 && lds_bytes <= 160 * 1024, "LDS");
};

struct WgPhGeom {
    int B, H, W, C;     // x extents
    int OH, OW;         // gy extents
    int PH, PW, K;
    int ni;             // images side by side: 1 (tiles of 64 columns) or 2 (32 columns each)
    int per;            // rows from one image to the next in the stack
    int passes;         // of a workgroup
    int nchunks, ncolt, nslices;
};

// One workgroup's run of rows: `blk` of the problem's `nblk` workgroups.
template <typename T, int NCOPY, int GR>
__device__ __forceinline__ void dwconv_wgrad_ph_body(const T* __restrict__ x, const T* __restrict__ gy,
                                                     float* __restrict__ part, const WgPhGeom& g, int blk, int nblk) {
    using Sh = WgPhShape<NCOPY, GR>;
    constexpr int NT = Sh::NT, CS = Sh::CS, CPW = Sh::CPW, XROW = Sh::XROW, XPL = Sh::XPL, GROW = Sh::GROW, GPL = Sh::GPL;
    constexpr bool EDGE = GR == 8;   // filters 16 and 17
    extern __shared__ uint32_t smem[];
    char* const xl = reinterpret_cast<char*>(smem);   // [buffer][channel][row][vector p][q] of T
    char* const gl = xl + 2 * Sh::XBUF;               // [buffer][channel][row][phase][q]

    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    int bid = xcd_remap(blk, nblk);
    const int sl = bid % g.nslices;
    bid /= g.nslices;
    const int ct = bid % g.ncolt, chunk = bid / g.ncolt;
    const int c0 = sl * CS, j0 = ct * (g.ni == 2 ? 32 : 64);
    const int V0 = chunk * g.passes * 8;                       // first row of the stack
    const int ngroups = (g.B + g.ni - 1) / g.ni;
    const int npasses = min(g.passes, ((ngroups - 1) * g.per + g.H - V0 + 7) >> 3);
    const int b_lo = max(V0 - 16, 0) / g.per;                  // first image (group) any row of the run lies in

    // ---- staging.  The wavefronts 0-3 stage x, 4-7 gy: a thread's item is (row of the pass, half of the q's, phase r,
    // 8-channel piece h), h fastest: columns 8q + r of its half, 4 of gy, 6 of x (the vectors p >= 8 are those of p - 8 one q
    // further).  Buffer loads whose offsets past the end read as zero without moving data: padding, tails, the rows between
    // images.
    const bool xs = wv < 4;
    const int ih = tid & 1, ir = (tid >> 1) & 7, ihalf = (tid >> 4) & 1, irow = (tid >> 5) & 7;
    constexpr uint32_t kNoCol = 0x40000000u, kNoRow = 0x80000000u;
    const uint32_t img_x = (uint32_t)(g.H * g.W * g.C), img_g = (uint32_t)(g.OH * g.OW * g.C);
    const int left = g.B - b_lo * g.ni, most = ((8 * g.passes + 16 + g.PH) / g.per + 2) * g.ni;
    const __amdgpu_buffer_rsrc_t xrsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<T*>(x + (long long)b_lo * g.ni * img_x), (short)0, (int)(min(left, most) * img_x * 2u), 0x00020000);
    const __amdgpu_buffer_rsrc_t grsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<T*>(gy + (long long)b_lo * g.ni * img_g), (short)0, (int)(min(left, most) * img_g * 2u), 0x00020000);
    const __amdgpu_buffer_rsrc_t srsrc = xs ? xrsrc : grsrc;
    auto bload = [&](const __amdgpu_buffer_rsrc_t& r, uint32_t off) {
        typedef unsigned v4u __attribute__((ext_vector_type(4)));
        const v4u v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0);
        return make_uint4(v.x, v.y, v.z, v.w);
    };
    const bool chok = c0 + 8 * ih < g.C;
    const int jc = j0 + (g.ni == 1 ? 32 * ihalf : 0) + ir;     // the item's first gy column
    auto column = [&](int j, int width, uint32_t img, bool ok) {   // byte offset of a column, or the marker
        return ok && chok && j >= 0 && j < width
                   ? ((g.ni == 2 ? (uint32_t)ihalf * img : 0u) + (uint32_t)(j * g.C + c0 + 8 * ih)) * 2u : kNoCol;
    };
    uint32_t col[6];
#pragma unroll
    for (int k = 0; k < 6; ++k)
        col[k] = xs ? column(jc + 8 * k - g.PW, g.W, img_x, true) : column(jc + 8 * k, g.OW, img_g, k < 4);
    const uint32_t row_bytes = (uint32_t)((xs ? g.W : g.OW) * g.C) * 2u, img_bytes = (xs ? img_x : img_g) * (uint32_t)g.ni * 2u;
    const int rows = xs ? g.H : g.OH;
    int sb, sr;   // image (group, from b_lo) and row of the item in the pass requested next
    {
        const int v = V0 + (xs ? 0 : g.PH) + irow;
        sb = v / g.per, sr = v - sb * g.per, sb -= b_lo;
    }
    uint4 buf[2][6];
    auto issue = [&](uint4 (&bf)[6], int pass) {   // called for the passes in order; those past the run read nothing
        const uint32_t r0 = pass < npasses && sr < rows && b_lo + sb < ngroups ? (uint32_t)sb * img_bytes + (uint32_t)sr * row_bytes : kNoRow;
#pragma unroll
        for (int k = 0; k < 6; ++k) bf[k] = bload(srsrc, r0 + col[k]);
        sr += 8;
        const bool wrap = sr >= g.per;   // (per >= 8)
        sr -= wrap ? g.per : 0, sb += wrap ? 1 : 0;
    };
    auto put = [](char* dst, uint32_t a0, uint32_t a1, uint32_t a2, uint32_t a3, uint32_t sel) {
        *reinterpret_cast<uint2*>(dst) = make_uint2(__builtin_amdgcn_perm(a1, a0, sel), __builtin_amdgcn_perm(a3, a2, sel));
    };
    // channel j of a piece is halfword j % 2 of dword j / 2
    auto dword = [](const uint4& u, int j) { return j < 2 ? u.x : j < 4 ? u.y : j < 6 ? u.z : u.w; };
    auto put_columns = [&](char* dst, const uint4 (&bf)[6], int j, int k) {   // columns k .. k + 3 of channel j
        put(dst, dword(bf[k], j), dword(bf[k + 1], j), dword(bf[k + 2], j), dword(bf[k + 3], j), j % 2 ? 0x07060302u : 0x05040100u);
    };
    // where an item goes: gy rows as they are, x rows 1 to NCOPY times (the first like gy)
    auto gy_dst = [&](char* base) { return base + 8 * ih * GPL + ih * Sh::HALF + irow * GROW + ir * 16 + ihalf * 8; };
    char* const xdst = xl + 8 * ih * XPL + ih * Sh::HALF + irow * XROW + ir * 16 + ihalf * 8;
    char* const sdst = xs ? xdst : gy_dst(gl);
    const int sbuf = xs ? Sh::XBUF : Sh::GBUF, spl = xs ? XPL : GPL;
    auto commit = [&](const uint4 (&bf)[6], int buffer, int j) { put_columns(sdst + buffer * sbuf + j * spl, bf, j, 0); };
    auto commit_copies = [&](const uint4 (&bf)[6], int buffer) {
        if (xs) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
                for (int c = 1; c < NCOPY; ++c) put_columns(xdst + buffer * Sh::XBUF + j * XPL + 128 * c, bf, j, c);
        }
    };
    auto lds_barrier = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    // the 16 gy rows above the run, 8 by each half of the wavefronts, go where pass 1 will: the nearer 8 into the second gy
    // buffer, the others, laid out like them, into the second x buffer
    static_assert(Sh::GBUF <= Sh::XBUF, "the rows above the run");
    {
        const int v = V0 + g.PH - 16 + (xs ? 0 : 8) + irow;
        const int b = v < 0 ? 0 : v / g.per, r = v - b * g.per;
        const uint32_t r0 = v >= 0 && r < g.OH && b < ngroups ? (uint32_t)(b - b_lo) * (img_g * (uint32_t)g.ni * 2u) + (uint32_t)(r * g.OW * g.C) * 2u : kNoRow;
#pragma unroll
        for (int k = 0; k < 4; ++k) buf[1][k] = bload(grsrc, r0 + column(jc + 8 * k, g.OW, img_g, true));
    }
    issue(buf[0], 0);
    {
        char* const dst = gy_dst(xs ? xl + Sh::XBUF : gl + Sh::GBUF);
#pragma unroll
        for (int j = 0; j < 8; ++j) put_columns(dst + j * GPL, buf[1], j, 0);
    }
    issue(buf[1], 1);
#pragma unroll
    for (int j = 0; j < 8; ++j) commit(buf[0], 0, j);
    commit_copies(buf[0], 0);
    issue(buf[0], 2);
    lds_barrier();

    // ---- operands.  A: lane = (v, phase of 4); B: lane = (row index n, phase of 4)
    const int ln = lane & 15, kg = lane >> 4;
    const int plane = wv * CPW, hoff = (plane >> 3) * Sh::HALF;
    const char* const xlane = xl + plane * XPL + hoff + (kg + min(ln, g.K - 1)) * 16;
    const char* const glane = gl + plane * GPL + hoff + (ln % GR) * GROW + kg * 16;
    auto read16 = [](const char* p) { return *reinterpret_cast<const uint4*>(p); };
    uint4 bop[CPW][2];
#pragma unroll
    for (int q = 0; q < CPW; ++q)
#pragma unroll
        for (int f = 0; f < 2; ++f)
            bop[q][f] = read16((ln < 8 ? xl + Sh::XBUF : gl + Sh::GBUF) + (plane + q) * GPL + hoff + (ln & 7) * GROW + (4 * f + kg) * 16);

    tz_f32x4 acc[CPW][8];
#pragma unroll
    for (int q = 0; q < CPW; ++q)
#pragma unroll
        for (int t = 0; t < 8; ++t) acc[q][t] = tz_f32x4{0.f, 0.f, 0.f, 0.f};

    // EDGE: column 16 and row 0 of the filter, which a product of 16 columns with the 16 rows before does not hold.
    // Column 16: products of the pass's 8 rows of x (index) with the 16 gy rows before the pass, and with its own 8:
    // u = m - n + 16 (n >= m: others lie beyond the filter) and m - n (n <= m).  Row 0: products of the phases r (index) with the
    // vectors p (0 .. 15 and 8 .. 23), four rows of x and gy at a time as the k groups: v = p - r.  A tap is a sum along a diagonal of both.
    tz_f32x4 before[EDGE ? CPW : 1], own[EDGE ? CPW : 1], row0[EDGE ? CPW : 1][2];
    if constexpr (EDGE) {
#pragma unroll
        for (int q = 0; q < CPW; ++q) before[q] = own[q] = row0[q][0] = row0[q][1] = tz_f32x4{0.f, 0.f, 0.f, 0.f};
    }
    // One pass from LDS buffer `buffer`, and the next one from registers into the other.
    auto pass_step = [&](int buffer, int pass) {
        const char* const xa = xlane + buffer * Sh::XBUF;
        const char* const ga = glane + buffer * Sh::GBUF;
        if constexpr (EDGE) {
            // a row at a time (blocks of two spill), its reads ahead of the products of the one before it
            uint4 a[2][2][CPW], n[CPW][2], ea[CPW][2], eb;
            auto read_row = [&](int row) {
#pragma unroll
                for (int f = 0; f < 2; ++f)
#pragma unroll
                    for (int q = 0; q < CPW; ++q) a[row % 2][f][q] = read16(xa + q * XPL + row * XROW + 64 * f);
            };
            // (the lane's part of these addresses is made in every pass: kept, they cost registers that others are spilled for,
            // [128,56,56,64] 48.8 us for 45.7)
            int here = lane;
            asm volatile("" : "+v"(here));
            const int en = here & 15, ek = here >> 4;
            const char* const xe = xl + plane * XPL + hoff + buffer * Sh::XBUF;
            const char* const ge = gl + plane * GPL + hoff + buffer * Sh::GBUF;
            auto read_row0 = [&](int i) {   // channel i % 2, rows 4 (i / 2) ..
                const int q = i % 2, r = 4 * (i / 2);
#pragma unroll
                for (int t = 0; t < 2; ++t) ea[0][t] = read16(xe + q * XPL + (r + ek) * XROW + (8 * t + en) * 16);
                eb = read16(ge + q * GPL + (r + ek) * GROW + (en & 7) * 16);
            };
#pragma unroll
            for (int q = 0; q < CPW; ++q)
#pragma unroll
                for (int f = 0; f < 2; ++f) {
                    n[q][f] = read16(ga + q * GPL + 64 * f);
                    ea[q][f] = read16(xe + q * XPL + (en & 7) * XROW + (16 + 4 * f + ek) * 16);
                }
            read_row(0);
#pragma unroll
            for (int q = 0; q < CPW; ++q)
#pragma unroll
                for (int f = 0; f < 2; ++f) {
                    before[q] = mfma16(ea[q][f], bop[q][f], before[q], T());
                    own[q] = mfma16(ea[q][f], n[q][f], own[q], T());
                }
#pragma unroll
            for (int row = 0; row < 8; ++row) {
                if (row < 7) read_row(row + 1);
                if (row < 4) read_row0(row);
                commit(buf[1 - buffer], 1 - buffer, row);
                __builtin_amdgcn_sched_barrier(0x7);
#pragma unroll
                for (int f = 0; f < 2; ++f)
#pragma unroll
                    for (int q = 0; q < CPW; ++q) acc[q][row] = mfma16(a[row % 2][f][q], bop[q][f], acc[q][row], T());
                if (row < 4) {
#pragma unroll
                    for (int t = 0; t < 2; ++t) row0[row % 2][t] = mfma16(eb, ea[0][t], row0[row % 2][t], T());
                }
                // the pass's gy row `row`, which index `row` of n holds
#pragma unroll
                for (int q = 0; q < CPW; ++q)
#pragma unroll
                    for (int f = 0; f < 2; ++f) {
                        uint4& b = bop[q][f];
                        b.x = ln == row ? n[q][f].x : b.x, b.y = ln == row ? n[q][f].y : b.y;
                        b.z = ln == row ? n[q][f].z : b.z, b.w = ln == row ? n[q][f].w : b.w;
                    }
                __builtin_amdgcn_sched_barrier(0x7);
                if (row == 5) commit_copies(buf[1 - buffer], 1 - buffer);
            }
        } else {
            // blocks of 2 rows, the reads of a block ahead of the products of the one before it (left to itself the compiler
            // requests the whole pass at once and spills)
            uint4 a[2][2][2][CPW], n[CPW][2];
            auto read_rows = [&](int blk) {
                if (2 * blk % GR == 0) {
#pragma unroll
                    for (int q = 0; q < CPW; ++q)
#pragma unroll
                        for (int f = 0; f < 2; ++f) n[q][f] = read16(ga + q * GPL + 2 * blk * GROW + 64 * f);
                }
#pragma unroll
                for (int r = 0; r < 2; ++r)
#pragma unroll
                    for (int f = 0; f < 2; ++f)
#pragma unroll
                        for (int q = 0; q < CPW; ++q) a[blk % 2][r][f][q] = read16(xa + q * XPL + (2 * blk + r) * XROW + 64 * f);
            };
            read_rows(0);
#pragma unroll
            for (int blk = 0; blk < 4; ++blk) {
                if (2 * blk % GR == 0) {
                    const bool enters = ln / GR == 2 * blk / GR;
#pragma unroll
                    for (int q = 0; q < CPW; ++q)
#pragma unroll
                        for (int f = 0; f < 2; ++f) {
                            uint4& b = bop[q][f];
                            b.x = enters ? n[q][f].x : b.x, b.y = enters ? n[q][f].y : b.y;
                            b.z = enters ? n[q][f].z : b.z, b.w = enters ? n[q][f].w : b.w;
                        }
                }
                if (blk < 3) read_rows(blk + 1);
                commit(buf[1 - buffer], 1 - buffer, 2 * blk), commit(buf[1 - buffer], 1 - buffer, 2 * blk + 1);
                __builtin_amdgcn_sched_barrier(0x7);
#pragma unroll
                for (int r = 0; r < 2; ++r)
#pragma unroll
                    for (int f = 0; f < 2; ++f)
#pragma unroll
                        for (int q = 0; q < CPW; ++q)
                            acc[q][2 * blk + r] = mfma16(a[blk % 2][r][f][q], bop[q][f], acc[q][2 * blk + r], T());
                __builtin_amdgcn_sched_barrier(0x7);
                if (blk == 1) commit_copies(buf[1 - buffer], 1 - buffer);
            }
        }
        issue(buf[1 - buffer], pass + 3);
        // in the next pass a row's index counts from 8 rows further
        auto ror8 = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf, true); };
#pragma unroll
        for (int q = 0; q < CPW; ++q)
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                uint4& b = bop[q][f];
                b = make_uint4(ror8(b.x), ror8(b.y), ror8(b.z), ror8(b.w));
            }
    };
    // Trips of 2 passes, left after the run's last pass (uniform).
    for (int p0 = 0; p0 < npasses; p0 += 2) {
#pragma unroll
        for (int jp = 0; jp < 2; ++jp) {
            const int pass = p0 + jp;
            lds_barrier();
            pass_step(jp, pass);
            if (pass + 1 >= npasses) {
                p0 = npasses;
                break;
            }
        }
    }
    // ---- the run's partial.  acc[t] holds the products of rows rho = t mod 8, its lane n the gy row rho - u with
    // u = t - n mod 16: rotated by 16 - t lanes they add up at lane -u mod 16.  Register r of a lane is v = 4 kg + r.
    tz_f32x4 tot[CPW];
#pragma unroll
    for (int q = 0; q < CPW; ++q) {
        tot[q] = acc[q][0];
#define PDW_ROT(t)                                                                                                     \
    for (int r = 0; r < 4; ++r)                                                                                        \
        tot[q][r] += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(acc[q][t][r]), 0x120 + 16 - t, 0xf, 0xf, true));
        PDW_ROT(1) PDW_ROT(2) PDW_ROT(3) PDW_ROT(4) PDW_ROT(5) PDW_ROT(6) PDW_ROT(7)
#undef PDW_ROT
    }
    lds_barrier();
    float* const ep = reinterpret_cast<float*>(smem);   // [tap][channel], 20 floats a tap
    constexpr int EPP = 20;
    const int u = EDGE ? 16 - ln : (16 - ln) & 15;   // (EDGE: the rows 16 .. 1 before)
#pragma unroll
    for (int q = 0; q < CPW; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int v = 4 * kg + r;
            if (u < g.K && v < g.K) ep[(u * g.K + v) * EPP + plane + q] = tot[q][r];
        }
    if constexpr (EDGE) {
        // sum of at_m[(lane + m) mod 16] over m < 8, at_m[n] being above[m] where n >= m and below[m] else; every lane group has it
        int here = tid;
        asm volatile("" : "+v"(here));   // (what follows from it is not worth registers during the passes)
        here &= 63;
        const int n = here & 15, group = here >> 4, first = n - 4 * (group & 1);   // m = 4 (group mod 2) + r
        auto diagonal = [&](const tz_f32x4& above, const tz_f32x4& below) {
            float t = first >= 0 ? above[0] : below[0];
#define PDW_ROT(r)                                                                             \
    t += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(first >= r ? above[r] : below[r]), 0x120 + 16 - r, 0xf, 0xf, true));
            PDW_ROT(1) PDW_ROT(2) PDW_ROT(3)
#undef PDW_ROT
            t = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(t), __float_as_int(t), 0x120 + 12, 0xa, 0xf, false));
            return t + __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(t), 0x401f));   // (lanes 16 apart)
        };
#pragma unroll
        for (int q = 0; q < CPW; ++q) {
            const float column = diagonal(before[q], own[q]), corner = diagonal(own[q], own[q]);   // (16 - lane, 16); lane 0: (0, 16)
            tz_f32x4 far;   // the vectors 16 .. 23 at the lanes 0 .. 7
#pragma unroll
            for (int r = 0; r < 4; ++r)
                far[r] = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(row0[q][1][r]), 0x128, 0xf, 0xf, true));
            const float row = diagonal(row0[q][0], far);   // (0, lane)
            const int tu = group == 0 ? 16 - n : 0, tv = group == 1 ? n : 16;
            if ((group < 2 || here == 32) && tu < g.K && tv < g.K) ep[(tu * g.K + tv) * EPP + plane + q] = group == 0 ? column : group == 1 ? row : corner;
        }
    }
    __syncthreads();
    float* const pc = part + (long long)(chunk * g.ncolt + ct) * g.K * g.K * g.C;
    for (int i = tid; i < g.K * g.K * (CS / 4); i += NT) {
        const int tap = i / (CS / 4), c4 = 4 * (i % (CS / 4));
        if (c0 + c4 < g.C) *reinterpret_cast<float4*>(pc + (long long)tap * g.C + c0 + c4) = *reinterpret_cast<const float4*>(ep + tap * EPP + c4);
    }
}

template <typename T, int NCOPY, int GR>
__global__ __launch_bounds__(512, 1) void dwconv_wgrad_ph_k(const T* __restrict__ x, const T* __restrict__ gy,
                                                            float* __restrict__ part, const WgPhGeom g) {
    dwconv_wgrad_ph_body<T, NCOPY, GR>(x, gy, part, g, blockIdx.x, gridDim.x);
}

// Two problems of the same filter size in one launch (the two scales of a block), the second problem's nblk1 workgroups first.
template <typename T, int NCOPY, int GR>
__global__ __launch_bounds__(512, 1) void dwconv_wgrad_ph_pair_k(const T* __restrict__ x0, const T* __restrict__ gy0,
                                                                 float* __restrict__ part0, const WgPhGeom g0,
                                                                 const T* __restrict__ x1, const T* __restrict__ gy1,
                                                                 float* __restrict__ part1, const WgPhGeom g1, int nblk1) {
    const bool second = (int)blockIdx.x < nblk1;
    const WgPhGeom g = second ? g1 : g0;
    dwconv_wgrad_ph_body<T, NCOPY, GR>(second ? x1 : x0, second ? gy1 : gy0, second ? part1 : part0, g,
                                       second ? blockIdx.x : blockIdx.x - nblk1, second ? nblk1 : gridDim.x - nblk1);
}

// ------------------------------------------------------------------------------------------------
// Host side

constexpr int kWgPhMaxK = 17;
constexpr int wgrad_ph_ncopy(int K) { return K <= 9 ? 2 : 3; }
constexpr int wgrad_ph_gr(int K) { return K <= 13 ? 4 : K <= 15 ? 2 : 8; }

struct WgPhPlan {
    bool ok = false;
    WgPhGeom g;
    long long per_chunk = 0, nblocks = 0;   // workgroups of a chunk (slices x column tiles), of the launch
    int total = 0;                          // passes of the whole stack
    int parts() const { return g.nchunks * g.ncolt; }
};

// Cuts the stack into `n` runs or a few less (equal ones but for the last); false: a run's images are beyond 32-bit offsets.
inline bool wgrad_ph_cut(WgPhPlan& p, int n) {
    WgPhGeom& g = p.g;
    g.passes = cdiv(p.total, n), g.nchunks = cdiv(p.total, g.passes);
    p.nblocks = p.per_chunk * g.nchunks;
    const long long images = ((8LL * g.passes + 16 + g.PH) / g.per + 2) * g.ni;
    const long long most = images < g.B ? images : g.B;
    const long long big = (long long)g.H * g.W > (long long)g.OH * g.OW ? (long long)g.H * g.W * g.C : (long long)g.OH * g.OW * g.C;
    return most * big <= 0x1fffffffLL && p.nblocks <= 0x7fffffffLL && (long long)g.nchunks * g.ncolt <= 0x7fffffffLL;
}

// Price of a run to the planners, us: start-up (16 gy rows, two round trips to memory, the partial), then passes of 8 rows.  (Of runs
// that share the chip with other problems; see the top for a chip full of them.  Beyond 15: training steps of [128,56,56,128],
// [16,40,40,256] and [26,106,105,80] with filter 17, us, at 2.1 437.2, 119.5, 280.6; 2.3 434.0, 119.7, 280.7; 2.5 432.8, 121.7, 282.1; 2.7 433.0,
// 121.6, 281.8.)
constexpr double kWgPhStart = 7.0;
inline double wgrad_ph_step(int K) { return K <= 9 ? 1.15 : K <= 15 ? 1.35 : 2.3; }
inline double wgrad_ph_run_cost(int K, int passes) { return kWgPhStart + wgrad_ph_step(K) * passes; }

// Covered: 16-bit types (the caller checks), C % 8 == 0, K <= 17, 16-byte aligned tensors.
inline WgPhPlan wgrad_ph_plan(int B, int H, int W, int C, int K, int PH, int PW) {
    WgPhPlan p;
    WgPhGeom& g = p.g;
    g.B = B, g.H = H, g.W = W, g.C = C, g.PH = PH, g.PW = PW, g.K = K;
    g.OH = H + 2 * PH - K + 1, g.OW = W + 2 * PW - K + 1;
    if (K < 1 || K > kWgPhMaxK || C % 8 != 0 || B < 1 || g.OH < 1 || g.OW < 1) return p;
    if ((long long)H * W * C > 0x1fffffffLL || (long long)g.OH * g.OW * C > 0x1fffffffLL) return p;
    g.ni = tz_wide_tile(B, g.OW) ? 1 : 2;
    // rows of one image never meet those of its neighbours: x row rho and gy row i do for -PH <= rho - i <= K-1-PH, OH = H + 2 PH - K + 1
    g.per = H + PH > g.OH ? H + PH : g.OH;
    if (g.per < 8) g.per = 8;
    g.ncolt = cdiv(g.OW, g.ni == 2 ? 32 : 64), g.nslices = cdiv(C, 16);
    const long long stack = (long long)(cdiv(B, g.ni) - 1) * g.per + H;
    if (stack + g.per + 64 > 0x7fffffffLL) return p;
    p.total = cdiv(stack, 8), p.per_chunk = (long long)g.ncolt * g.nslices;
    // runs: as many as fill 256 compute units 1..4 times, whichever is estimated to end first (a partial costs its bytes twice)
    int best = 0;
    double best_cost = 0;
    for (int rounds = 1; rounds <= 4; ++rounds) {
        const long long want = 256LL * rounds / p.per_chunk;
        const int n = want < 1 ? 1 : want > p.total ? p.total : (int)want;
        if (!wgrad_ph_cut(p, n)) continue;
        const double cost = cdiv(p.nblocks, 256) * wgrad_ph_run_cost(K, g.passes) + 8e-6 * g.nchunks * g.ncolt * K * K * C / 4.0;
        if (best == 0 || cost < best_cost) best = n, best_cost = cost;
    }
    if (best == 0) {   // large images: runs as short as their offsets need
        if (!wgrad_ph_cut(p, p.total)) return p;
        best = p.total;
    }
    p.ok = wgrad_ph_cut(p, best);
    return p;
}

template <typename T, int NCOPY, int GR>
static int launch_wgrad_ph(const WgPhPlan& p, const void* x, const void* gy, void* ws, hipStream_t s) {
    using Sh = WgPhShape<NCOPY, GR>;
    auto kern = dwconv_wgrad_ph_k<T, NCOPY, GR>;
    static std::once_flag attr_once;
    std::call_once(attr_once, [&] { (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); });
    hipLaunchKernelGGL(kern, dim3((unsigned)p.nblocks), dim3(Sh::NT), Sh::lds_bytes, s, (const T*)x, (const T*)gy, (float*)ws, p.g);
    return check_launch("dwconv_wgrad_ph");
}

template <typename T, int NCOPY, int GR>
static int launch_wgrad_ph_pair(const WgPhPlan& p0, const void* x0, const void* gy0, void* ws0, const WgPhPlan& p1,
                                const void* x1, const void* gy1, void* ws1, hipStream_t s) {
    using Sh = WgPhShape<NCOPY, GR>;
    auto kern = dwconv_wgrad_ph_pair_k<T, NCOPY, GR>;
    static std::once_flag attr_once;
    std::call_once(attr_once, [&] { (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); });
    if (p0.nblocks + p1.nblocks > 0x7fffffffLL) return -1;
    hipLaunchKernelGGL(kern, dim3((unsigned)(p0.nblocks + p1.nblocks)), dim3(Sh::NT), Sh::lds_bytes, s, (const T*)x0, (const T*)gy0,
                       (float*)ws0, p0.g, (const T*)x1, (const T*)gy1, (float*)ws1, p1.g, (int)p1.nblocks);
    return check_launch("dwconv_wgrad_ph_pair");
}

}  // namespace pdw
