// Depthwise convolution in fp32 on the fp32 matrix cores: forward and input gradient, stride 1, dilation 1, odd square
// filters 3 .. 17 (the input gradient is the same kernel on gy with the rotated filter and padding k-1-p).
//
// The block-Toeplitz product of dwconv_tz.h on v_mfma_f32_16x16x4_f32: for one channel m = the 16 outputs of a 4 x 4 patch,
// n = 16 patches four columns apart (in NI = 16 / NPC images), k = 4 consecutive columns of one window row.
//     A[(di,dj)][(r, 4j+g)] = w[r - di][4j + g - dj]     IC * JB of them (IC = K+3 rows, JB column blocks), kept in registers as far as
//                                                       two workgroups of a compute unit leave room (f32t_kept), else read from LDS
//     B[(r, 4j+g)][n]       = window[r][4n + 4j + g]      64 consecutive floats of a staged row: one conflict-free LDS read
// A window row belongs to up to PER = ceil(IC/4) patch rows, whose accumulators are all live: a B operand is read once and
// feeds PER products of 32 cycles each, so the matrix pipe is what bounds the kernel (LDS is under 10 % busy), a row
// is dead after its step, and the window in LDS is two groups of four rows whatever the filter (20 KB).  Vector instructions do
// not overlap with fp32 products (measured with products by one wavefront of a SIMD and additions by another: 124 and 172 us
// alone, 289 together), so what the staging computes per thread is added to the products' time: offsets are those of a
// workgroup plus a scalar row offset wherever all rows of a group exist, and the accumulators rotate by the products' own
// addend operand.  A step in which all accumulators are live runs without a branch, the products of a row alternating
// between them.
//
// A workgroup (8 wavefronts, one channel each) owns a band of output rows x 4 NPC columns x NI images of 8 channels.  A step is
// four window rows: the wavefronts multiply them, commit the next four from registers (16 bytes = 4 channels of a pixel,
// written channel-major), request the rows two steps ahead, and store the patch row that the previous step finished
// (through a pixel-major tile in LDS, 16 bytes a thread).  One barrier a step; wavefronts 0-3 multiply first and 4-7 last, so
// that of a SIMD's two wavefronts one always feeds the matrix pipe.
//
// Measured at [32,56,56,64], filter 13: 35.1 us (36.7 with the conditions per thread and per product; the products alone 27 at
// the clock that they leave, vector-ALU kernel (dwconv_tiled.h) 77); [3,57,61,100] filter 15 14.9 (15.9); [8,112,112,48] filter
// 17 38.3 (41.0); [1,5,90,36] filter 17 8.5 (9.7).
//
// ADD: the input gradient of a tensor that was also average-pooled to (AH, AW): y += the pool's gradient, from the one bin of
// a pixel where the pool halved both extents (1), gathered from the at most 2 x 2 bins that a pixel lies in (2).
#pragma once
#include <mutex>

#include "common.h"
#include "kernels.h"
#include "tile_common.h"

namespace pdw {

// Column blocks of A operands that stay in registers, all of them or what leaves a wavefront 128 registers, so that two workgroups share a
// compute unit; the others are read again from the filter table in LDS for every product (a fifth of its rate).  us, all in registers and one
// workgroup a unit -> this: both scales of [32,56,56,64] filter 13 50.5 -> 45.5, [22,72,73,32] filter 13 36.6 -> 32.2, [3,57,61,100]
// filter 15 24.2 -> 18.2, [16,56,56,64] filter 15 38.9 -> 33.3, [24,36,36,100] filter 17 57.0 -> 50.7, [2,20,20,32] filter 15 9.0 -> 8.5.  With the pooled
// gradient added (ADD > 0), which the planner cuts into one workgroup a unit, all stay ([32,56,56,64] filter 13 38.3, 39.2 with three
// blocks kept, [24,36,36,100] filter 17 35.8 and 36.6), and in launches of no more than that whose bands are of three patch rows or more (ADD = -1),
// where reading operands again outweighs the longer start-up: with two or three blocks kept -> all, by the rows of a band, 12: [77,10,10,80]
// filter 15 12.9 -> 12.4, [40,25,25,312] 16.4 -> 15.7, [3,106,107,112] filter 17 17.4 -> 17.0; 16: [21,31,32,276] filter 17 23.1 -> 22.3; 24: [7,21,20,440]
// filter 13 10.8 -> 10.5, [6,45,60,152] filter 15 26.5 -> 25.3; 48: [19,45,49,92] 16.9 -> 15.9; 56: [32,56,56,64] filter 13 39.7 -> 38.7, [1,106,106,496]
// filter 17 22.3 -> 21.2 (25 such launches, all of them faster); 8: [34,16,16,60] filter 17 10.0 and 11.0; 4: [8,12,16,252] filter 13 8.0 and 8.4.
template <int K, int ADD>
constexpr int f32t_kept() {
    return ADD != 0 || K <= 11 ? (K + 6) / 4 : K == 13 ? 3 : 2;
}

template <int K, int NPC, int ADD = 0>
struct F32Shape {
    static constexpr int NT = 512, CS = 8;
    static constexpr int IC = K + 3, JB = (IC + 3) / 4, PER = (IC + 3) / 4, NI = 16 / NPC, TW = 4 * NPC;
    static constexpr int WCOLS = 4 * (NPC - 1) + 4 * JB;          // window columns of an image
    static constexpr int RP = 4 * WCOLS;                           // bytes per window row of a channel
    // bytes per channel plane (8 rows): images of an operand read and channel quads of a staging write on other banks
    static constexpr int plane() {
        int p = 8 * RP;
        const int want = NI == 1 ? 32 : NI == 2 ? 16 : 8, mod = NI == 1 ? 64 : 32;
        while (p % mod != want) p += 8;
        return p;
    }
    static constexpr int CHP = plane();
    static constexpr int OROWP = TW * 32 + NPC * 4;                // result tile: row pitch (4 bytes more every 4 pixels)
    static constexpr int OLB = NI * 4 * OROWP;
    static constexpr int WTH = K + 6, WTW = 4 * JB + 4;            // zero-bordered filter table of a channel
    static constexpr bool STREAM = f32t_kept<K, ADD>() < JB;       // the table stays, behind the result tiles
    static constexpr int TAB = (CS * WTH * WTW * 4 + 15) / 16 * 16, OTB = (2 * OLB + 15) / 16 * 16;
    static constexpr int R2B = STREAM ? OTB + TAB : OTB > TAB ? OTB : TAB;
    static constexpr size_t lds_bytes = (size_t)NI * CS * CHP + R2B;
    static constexpr int NLD = (4 * NI * WCOLS * 2 + NT - 1) / NT; // staging items per thread and step
    static_assert(lds_bytes <= 80 * 1024 && NLD <= 2, "sizes");
};

struct F32Geom {
    int B, H, W, C, OH, OW, PH, PW, BR, nbands, ncolt, nslices, flip, AH, AW;
};

template <int K, int NPC, int ADD>
__device__ __forceinline__ void dwconv_f32_body(const float* __restrict__ x, const float* __restrict__ w,
                                                const float* __restrict__ add, float* __restrict__ y, const F32Geom& g, int blk,
                                                int nblk) {
    using Sh = F32Shape<K, NPC, ADD>;
    constexpr int NT = Sh::NT, IC = Sh::IC, JB = Sh::JB, PER = Sh::PER, NI = Sh::NI, TW = Sh::TW, RP = Sh::RP, CHP = Sh::CHP;
    constexpr int JR = f32t_kept<K, ADD>();
    constexpr int OROWP = Sh::OROWP, OLB = Sh::OLB, WTH = Sh::WTH, WTW = Sh::WTW, NLD = Sh::NLD, WCOLS = Sh::WCOLS, CS = Sh::CS;
    typedef float f4 __attribute__((ext_vector_type(4)));
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    extern __shared__ uint32_t smem[];
    char* const xl = reinterpret_cast<char*>(smem);
    char* const r2 = xl + NI * CS * CHP;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    int bid = xcd_remap(blk, nblk);
    const int sl = bid % g.nslices;
    bid /= g.nslices;
    const int ct = bid % g.ncolt;
    bid /= g.ncolt;
    const int band = bid % g.nbands, b0 = bid / g.nbands * NI;
    const int c0 = sl * CS, ocol0 = ct * TW, orow0 = band * g.BR;
    const int rows_valid = min(g.BR, g.OH - orow0), cols_valid = min(TW, g.OW - ocol0);
    const int npr = (rows_valid + 3) >> 2, nsteps = npr + PER - 1;   // patch rows; groups of four window rows
    const long long img_in = (long long)g.H * g.W * g.C, img_out = (long long)g.OH * g.OW * g.C;

    // ---- filter slice to registers (before the window's loads), then to the zero-bordered table
    constexpr int NWL = (K * K * 2 + NT - 1) / NT;
    f4 wval[NWL];
#pragma unroll
    for (int i = 0; i < NWL; ++i) {
        const int idx = min(tid + i * NT, K * K * 2 - 1);
        wval[i] = *reinterpret_cast<const f4*>(w + (idx >> 1) * g.C + min(c0 + 4 * (idx & 1), g.C - 4));
    }
    // ---- staging: offsets past the descriptor's end (images beyond the batch, the markers) read as zero
    constexpr uint32_t kNoRow = 0x80000000u;
    const __amdgpu_buffer_rsrc_t xrsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(x + (long long)b0 * img_in), (short)0, (int)(min(NI, g.B - b0) * img_in * 4), 0x00020000);
    uint32_t xoff[NLD];   // bytes from the group's first row, or kNoRow
    int irow[NLD], idst[NLD];
#pragma unroll
    for (int l = 0; l < NLD; ++l) {
        const int idx = tid + l * NT, q = idx & 1, col = (idx >> 1) % WCOLS, img = (idx >> 1) / WCOLS % NI;
        irow[l] = (idx >> 1) / WCOLS / NI;
        const int ic = ocol0 - g.PW + col;
        const bool ok = irow[l] < 4 && c0 + 4 * q < g.C && ic >= 0 && ic < g.W;
        xoff[l] = ok ? ((uint32_t)img * (uint32_t)img_in + (uint32_t)((irow[l] * g.W + ic) * g.C + c0 + 4 * q)) * 4u : kNoRow;
        idst[l] = (img * CS + 4 * q) * CHP + (irow[l] & 3) * RP + col * 4;
    }
    f4 buf[2][NLD];
    auto issue = [&](f4 (&bf)[NLD], int s) {
        const int ir0 = orow0 - g.PH + 4 * s, row_at = ir0 * g.W * g.C * 4;
        uint32_t xo[NLD];
        int so = row_at;
#pragma unroll
        for (int l = 0; l < NLD; ++l) xo[l] = xoff[l];
        if (s >= nsteps || ir0 < 0 || ir0 + 3 >= g.H) {   // (uniform; where all four rows exist, nothing to compute per thread)
            so = 0;
#pragma unroll
            for (int l = 0; l < NLD; ++l) {
                const bool ok = (int)xoff[l] >= 0 && s < nsteps && (unsigned)(ir0 + irow[l]) < (unsigned)g.H;
                xo[l] = ok ? xoff[l] + (uint32_t)row_at : kNoRow;
            }
        }
#pragma unroll
        for (int l = 0; l < NLD; ++l) bf[l] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(xrsrc, (int)xo[l], so, 0));
    };
    auto commit = [&](const f4 (&bf)[NLD], int half) {   // half of the window: 0 or 1
#pragma unroll
        for (int l = 0; l < NLD; ++l) {
            if (wv * 64 + l * NT < 8 * NI * WCOLS && ((l + 1) * NT <= 8 * NI * WCOLS || irow[l] < 4)) {
                const float e0 = bf[l].x, e1 = bf[l].y, e2 = bf[l].z, e3 = bf[l].w;
                char* d = xl + idst[l] + half * 4 * RP;
                *reinterpret_cast<float*>(d) = e0;
                *reinterpret_cast<float*>(d + CHP) = e1;
                *reinterpret_cast<float*>(d + 2 * CHP) = e2;
                *reinterpret_cast<float*>(d + 3 * CHP) = e3;
            }
        }
    };
    issue(buf[0], 0);
    issue(buf[1], 1);
    auto lds_barrier = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    float* const wt = reinterpret_cast<float*>(r2 + (Sh::STREAM ? Sh::OTB : 0));   // [channel][3 + u][3 + v]
    for (int i = tid; i < CS * WTH * WTW / 4; i += NT) reinterpret_cast<f4*>(wt)[i] = f4{0.f, 0.f, 0.f, 0.f};
    lds_barrier();
#pragma unroll
    for (int i = 0; i < NWL; ++i) {
        const int idx = tid + i * NT, q = idx & 1, uv = idx >> 1, u = uv / K, v = uv - u * K;
        if (idx < K * K * 2 && c0 + 4 * q < g.C) {
            const int uu = g.flip ? K - 1 - u : u, vv = g.flip ? K - 1 - v : v;
            float* wp = wt + (4 * q * WTH + 3 + uu) * WTW + 3 + vv;
            const float e0 = wval[i].x, e1 = wval[i].y, e2 = wval[i].z, e3 = wval[i].w;
            wp[0] = e0, wp[WTH * WTW] = e1, wp[2 * WTH * WTW] = e2, wp[3 * WTH * WTW] = e3;
        }
    }
    commit(buf[0], 0);
    issue(buf[0], 2);
    lds_barrier();
    // ---- this wavefront's A operands
    const int ln = lane & 15, kg = lane >> 4;
    float A[IC][JR];
    const float* const wp = wt + (wv * WTH + 3 - (ln >> 2)) * WTW + 3 + kg - (ln & 3);
#pragma unroll
    for (int r = 0; r < IC; ++r)
#pragma unroll
        for (int j = 0; j < JR; ++j) A[r][j] = wp[r * WTW + 4 * j];
    if constexpr (!Sh::STREAM) lds_barrier();   // (the table's space becomes the result tiles)
    uint32_t wb[2] = {0, 0};   // rows 0 and 8 of this lane's table (as xb below)
    if constexpr (Sh::STREAM) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            wb[i] = (uint32_t)(reinterpret_cast<const char*>(wp) - xl) + (uint32_t)(8 * i * WTW * 4);
            asm("" : "+v"(wb[i]));
        }
    }
    auto weight = [&](int row, int j) { return *reinterpret_cast<const float*>(xl + wb[row / 8 < 2 ? row / 8 : 1] + ((row - (row < 8 ? 0 : 8)) * WTW + 4 * j) * 4); };
    const int pimg = ln / NPC, pc = ln % NPC;
    // Rows 0 .. 7 of the window at a lane, in three registers: as offsets from one they are out of a paired read's reach, and
    // each read would add its own (vector instructions do not overlap with fp32 products: 124 us of products and 172 us of
    // additions by another wavefront take 289 us).
    uint32_t xb[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        xb[i] = (uint32_t)((pimg * CS + wv) * CHP + (4 * pc + kg) * 4 + 3 * i * RP);
        asm("" : "+v"(xb[i]));
    }
    // result of a lane: patch ln, row kg, columns 4 pc .. + 3 (the four registers)
    char* const olw = r2 + (pimg * 4 + kg) * OROWP + pc * (4 * 32 + 4) + wv * 4;
    const int sq = tid & 1, scol = (tid >> 1) % TW, srow = (tid >> 1) / TW % 4, simg = (tid >> 1) / TW / 4;
    const bool s_ok = scol < cols_valid && c0 + 4 * sq < g.C;
    const char* const olr = r2 + (simg * 4 + srow) * OROWP + scol * 32 + (scol >> 2) * 4 + 16 * sq;
    const __amdgpu_buffer_rsrc_t yrsrc = __builtin_amdgcn_make_buffer_rsrc(
        y + (long long)b0 * img_out, (short)0, (int)(min(NI, g.B - b0) * img_out * 4), 0x00020000);
    const uint32_t yoff = s_ok ? ((uint32_t)simg * (uint32_t)img_out + (uint32_t)((srow * g.OW + ocol0 + scol) * g.C + c0 + 4 * sq)) * 4u : kNoRow;
    __amdgpu_buffer_rsrc_t arsrc = xrsrc;
    int jb0 = 0;
    uint32_t aoff = 0;
    float wj0 = 0.f, wj1 = 0.f, wi0 = 0.f, wi1 = 0.f;
    f4 addv[ADD == 2 ? 4 : 1];
    float* const bins = reinterpret_cast<float*>(xl + Sh::lds_bytes);   // ADD 2: (byte offset of the first bin, both weights) of the band's rows
    if constexpr (ADD > 0) {
        arsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(add + (long long)b0 * g.AH * g.AW * g.C), (short)0,
                                                  (int)((long long)min(NI, g.B - b0) * g.AH * g.AW * g.C * 4), 0x00020000);
        if constexpr (ADD == 2) {
            // (read behind the barrier before the first add_fetch)
            for (int i = tid; i < rows_valid; i += NT) {
                int b;
                float w0, w1;
                pool_bins(orow0 + i, g.OH, g.AH, b, w0, w1);
                bins[4 * i] = __builtin_bit_cast(float, (uint32_t)(b * g.AW * g.C) * 4u), bins[4 * i + 1] = w0, bins[4 * i + 2] = w1;
            }
            pool_bins(min(ocol0 + scol, g.OW - 1), g.OW, g.AW, jb0, wj0, wj1);
            aoff = ((uint32_t)(simg * g.AH * g.AW + jb0) * (uint32_t)g.C + (uint32_t)(c0 + 4 * sq)) * 4u;
        } else aoff = s_ok ? ((uint32_t)((simg * g.AH + (srow >> 1)) * g.AW + ((ocol0 + scol) >> 1)) * (uint32_t)g.C + (uint32_t)(c0 + 4 * sq)) * 4u : kNoRow;
    }
    auto add_fetch = [&](int pr) {   // the bins of patch row pr's pixels
        if constexpr (ADD == 1) {
            uint32_t o = aoff;
            if (pr < 0 || 4 * pr + 3 >= rows_valid) o = pr >= 0 && 4 * pr + srow < rows_valid ? o : kNoRow;
            // (below the band no scalar offset either: it could lie past the descriptor's end, from which the range check subtracts it)
            const int at = pr >= 0 && 4 * pr < rows_valid ? ((orow0 + 4 * pr) >> 1) * g.AW * g.C * 4 : 0;
            addv[0] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(arsrc, (int)o, at, 0));
        } else if constexpr (ADD == 2) {
            // (from the table: found anew for every row they were 600 cycles a step that no product covers; us: [3,57,61,100] filter 15 21.4 ->
            // 19.2, [22,72,73,32] filter 13 33.4 -> 29.2, [8,47,48,128] filter 17 33.0 -> 29.0, [8,27,31,40] filter 11 11.7 -> 9.2)
            const float4 bin = *reinterpret_cast<const float4*>(bins + 4 * min(max(4 * pr + srow, 0), rows_valid - 1));
            wi0 = bin.y, wi1 = bin.z;
            const bool ok = s_ok && pr >= 0 && 4 * pr + srow < rows_valid;
            const uint32_t o = aoff + __builtin_bit_cast(uint32_t, bin.x);
            const uint32_t dx = (uint32_t)g.C * 4u, dy = (uint32_t)(g.AW * g.C) * 4u;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const bool in = ok && ((t & 1) == 0 || wj1 != 0.f) && ((t & 2) == 0 || wi1 != 0.f);
                const uint32_t off = in ? o + (t & 1 ? dx : 0u) + (t & 2 ? dy : 0u) : kNoRow;
                addv[t] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(arsrc, (int)off, 0, 0));
            }
        }
    };
    auto store = [&](int pr) {   // patch row pr from its tile (outside the band: nothing)
        const char* src = olr + (pr & 1) * OLB;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = *reinterpret_cast<const float*>(src + 4 * e);
        if constexpr (ADD == 1) {
            const float a0 = addv[0].x, a1 = addv[0].y, a2 = addv[0].z, a3 = addv[0].w;
            v[0] += 0.25f * a0, v[1] += 0.25f * a1, v[2] += 0.25f * a2, v[3] += 0.25f * a3;
        } else if constexpr (ADD == 2) {
            const float k00 = wi0 * wj0, k01 = wi0 * wj1, k10 = wi1 * wj0, k11 = wi1 * wj1;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                v[e] += fmaf(k11, addv[3][e], fmaf(k10, addv[2][e], fmaf(k01, addv[1][e], k00 * addv[0][e])));
        }
        uint32_t o = yoff;
        if (pr < 0 || 4 * pr + 3 >= rows_valid) o = pr >= 0 && 4 * pr + srow < rows_valid ? o : kNoRow;   // (uniform)
        const int at = pr >= 0 ? (orow0 + 4 * pr) * g.OW * g.C * 4 : 0;   // (no scalar offset in a 16-byte store: see dwconv_tz.h)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, f4{v[0], v[1], v[2], v[3]}), yrsrc, (int)(o + (uint32_t)at), 0, 0);
    };
    // acc[q]: the patch row whose q-th group of window rows was multiplied last.  Step s multiplies window rows 4 s .. 4 s + 3
    // for patch rows s - q and finishes patch row s - PER + 1; every patch row moves one accumulator up in its first product.
    f4 acc[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) acc[q] = f4{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](int half, int s) {
        auto fetch = [&](float (&bv)[JB], int r) {
            const int row = half * 4 + r;
#pragma unroll
            for (int j = 0; j < JB; ++j) bv[j] = *reinterpret_cast<const float*>(xl + xb[row / 3] + row % 3 * RP + 16 * j);
        };
        if (s >= PER - 1 && s < npr) {   // (uniform) all of them: row by row, the next row's operands read meanwhile
            float bv[2][JB], av[2][PER];   // (av: of the column blocks that are not kept, a block ahead)
            fetch(bv[0], 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (r < 3) fetch(bv[(r + 1) & 1], r + 1);
#pragma unroll
                for (int j = 0; j < JB; ++j) {
                    if (j + 1 >= JR && j + 1 < JB) {
#pragma unroll
                        for (int q = PER - 1; q >= 0; --q)
                            if (4 * q + r < IC) av[(j + 1) & 1][q] = weight(4 * q + r, j + 1);
                    }
#pragma unroll
                    for (int q = PER - 1; q >= 0; --q) {
                        if (4 * q + r >= IC) continue;
                        const f4 c = r == 0 && j == 0 ? (q > 0 ? acc[q > 0 ? q - 1 : 0] : f4{0.f, 0.f, 0.f, 0.f}) : acc[q];
                        const float w = j < JR ? A[4 * q + r < IC ? 4 * q + r : 0][j < JR ? j : 0] : av[j & 1][q];
                        acc[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(w, bv[r & 1][j], c, 0, 0, 0);
                    }
                }
            }
        } else {   // the first and last patch rows: one after the other
#pragma unroll
            for (int q = PER - 1; q >= 0; --q) {
                if (s < q || s - q >= npr) continue;   // (uniform)
                f4 a = q > 0 ? acc[q > 0 ? q - 1 : 0] : f4{0.f, 0.f, 0.f, 0.f};
                float bv[2][JB], av[2][JB > JR ? JB - JR : 1];
                auto weights = [&](float (&d)[JB > JR ? JB - JR : 1], int r) {
#pragma unroll
                    for (int j = JR; j < JB; ++j)
                        if (4 * q + r < IC) d[j - JR] = weight(4 * q + r, j);
                };
                fetch(bv[0], 0);
                weights(av[0], 0);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (4 * q + r >= IC) continue;
                    if (r < 3) fetch(bv[(r + 1) & 1], r + 1), weights(av[(r + 1) & 1], r + 1);
#pragma unroll
                    for (int j = 0; j < JB; ++j) {
                        const float w = j < JR ? A[4 * q + r < IC ? 4 * q + r : 0][j < JR ? j : 0] : av[r & 1][j >= JR ? j - JR : 0];
                        a = __builtin_amdgcn_mfma_f32_16x16x4f32(w, bv[r & 1][j], a, 0, 0, 0);
                    }
                }
                acc[q] = a;
            }
        }
        const int pr = s - PER + 1;
        if (pr >= 0 && pr < npr) {
            char* d = olw + (pr & 1) * OLB;
            const float e0 = acc[PER - 1].x, e1 = acc[PER - 1].y, e2 = acc[PER - 1].z, e3 = acc[PER - 1].w;
            *reinterpret_cast<float*>(d) = e0;
            *reinterpret_cast<float*>(d + 32) = e1;
            *reinterpret_cast<float*>(d + 64) = e2;
            *reinterpret_cast<float*>(d + 96) = e3;
        }
    };
    auto step = [&](f4 (&bf)[NLD], int half, int s) {   // bf: holds the rows of step s + 1
        lds_barrier();   // the rows of step s are in place, and everybody is done with those of s - 1
        if (wv < 4 && s < nsteps) compute(half, s);
        store(s - PER);                      // (finished by step s - 1)
        add_fetch(s - PER + 1);              // for the next step's store
        commit(bf, half ^ 1);
        issue(bf, s + 3);
        if (wv >= 4 && s < nsteps) compute(half, s);
    };
    if constexpr (ADD == 2) lds_barrier();   // (the bins)
    add_fetch(-1);
    // (the two buffers by name and no way out between them: the compiler can then tell which requests are the newest, and a
    // commit waits for its own alone)
    int s = 0;
    do {
        step(buf[1], 0, s);
        step(buf[0], 1, s + 1);
        s += 2;
    } while (s < nsteps);
    lds_barrier();
    if (s == nsteps) store(nsteps - PER);   // (else the step past the last did)
}

// Register bound: two workgroups on a compute unit where the filter's operands leave room, so that one's start-up
// overlaps the other's products.
template <int K, int ADD>
constexpr int f32t_waves() {
    return (K >= 13 && ADD == 0) || (K + 3) * ((K + 6) / 4) <= (ADD ? 36 : 56) ? 4 : 2;
}

template <int K, int NPC, int ADD>
__global__ __launch_bounds__(512, (f32t_waves<K, ADD>())) void dwconv_f32t_k(const float* __restrict__ x, const float* __restrict__ w,
                                                                     const float* __restrict__ add, float* __restrict__ y,
                                                                     const F32Geom g) {
    dwconv_f32_body<K, NPC, ADD>(x, w, add, y, g, blockIdx.x, gridDim.x);
}

// ------------------------------------------------------------------------------------------------
// Host side

// Patches side by side (16, or 8 or 4 in two or four images): the width whose padding of (columns x images) is smallest.
inline int f32t_npc(int B, int OW) {
    int best = 16;
    long long least = -1;
    for (int npc = 16; npc >= 4; npc /= 2) {
        const int tw = 4 * npc, ni = 16 / npc;
        const long long pad = (long long)cdiv(OW, tw) * tw * cdiv(B, ni) * ni;
        if (least < 0 || pad < least) least = pad, best = npc;
    }
    return best;
}

// Band height: the fewest cycles for rounds of workgroups over 256 compute units (products of the band; start-up and the
// window's first rows, which two workgroups of a unit overlap).
template <int K>
int f32t_band(long long per_band, int OH, bool add) {
    constexpr int NA = (K + 3) * ((K + 6) / 4);
    if (const char* e = tune_env("PDW_F32_BR")) return atoi(e);
    int best = 4;
    double cost = -1;
    for (int br = 4; br <= (OH + 3) / 4 * 4; br += 4) {
        const long long wgs = per_band * cdiv(OH, br);
        const double c = (double)cdiv(wgs, 256) * (br / 4) * NA * 64 + (double)cdiv(wgs, f32t_waves<K, 0>() == 4 && (K < 13 || !add) ? 512 : 256) * 9000;
        if (cost < 0 || c <= cost) cost = c, best = br;
    }
    return best;
}

// Where the vector-ALU kernel (dwconv_tiled.h) stays, unless the pooled gradient rides here (which saves a pass over y):
// - filters 3 and 7 once the tensor is more than a round of workgroups ([40,14,14,256] filter 7: 14.5 us here, 11.9 there), whose
//   values that are not finite reach no further than the filter there; 5 there unless the images fill the tiles
//   ([40,70,70,64]: 30 here, 45 there);
// - filters 9 and 11 on images that leave half of a tile's columns empty ([100,7,7,1152] filter 9: 61 here, 46 there).
template <int K>
bool f32t_pays(long long outputs, int OW, int npc, bool add) {
    if (K >= 13 || add) return true;
    const int tw = 4 * npc, filled = OW * 100 / (cdiv(OW, tw) * tw);   // per cent of the columns
    if (K <= 7 && outputs <= 350000) return true;
    return K == 5 ? filled >= 82 : K > 7 && filled >= 55;
}

// false: not covered
template <int K>
bool f32t_geom(F32Geom& g, int& npc, long long& nblocks, int B, int H, int W, int C, int PH, int PW, bool flip, bool add = false) {
    g = F32Geom{B, H, W, C, H + 2 * PH - K + 1, W + 2 * PW - K + 1, PH, PW, 0, 0, 0, 0, flip ? 1 : 0, 0, 0};
    if (g.OH < 1 || g.OW < 1 || C % 4 != 0 || B < 1) return false;
    npc = f32t_npc(B, g.OW);
    const int ni = 16 / npc;
    if ((long long)H * W * C * ni > 0x0fffffffLL || (long long)g.OH * g.OW * C * ni > 0x0fffffffLL) return false;
    g.ncolt = cdiv(g.OW, 4 * npc), g.nslices = cdiv(C, 8);
    const long long per_band = (long long)cdiv(B, ni) * g.ncolt * g.nslices;
    g.BR = f32t_band<K>(per_band, g.OH, add), g.nbands = cdiv(g.OH, g.BR);
    nblocks = per_band * g.nbands;
    return nblocks <= 0x7fffffffLL;
}

// -1: not covered.  add (optional): [B, AH, AW, C], AH <= OH, AW <= OW.
template <int K>
int launch_f32t(const void* x, const void* w, const void* add, void* y, int B, int H, int W, int C, int PH, int PW, bool flip,
                int AH, int AW, hipStream_t s) {
    F32Geom g;
    int npc;
    long long nblocks;
    if (!f32t_geom<K>(g, npc, nblocks, B, H, W, C, PH, PW, flip, add != nullptr)) return -1;
    if (!f32t_pays<K>((long long)B * g.OH * g.OW * C, g.OW, npc, add != nullptr)) return -1;
    for (const void* p : {x, w, (const void*)y, add})
        if (reinterpret_cast<uintptr_t>(p) & 15) return -1;
    if (add && (AH > g.OH || AW > g.OW || AH < 1 || AW < 1)) return -1;
    g.AH = AH, g.AW = AW;
#define PDW_F32T(NPC, A)                                                                                                   \
    {                                                                                                                      \
        auto kern = dwconv_f32t_k<K, NPC, A>;                                                                              \
        static std::once_flag once;                                                                                        \
        std::call_once(once, [&] { (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); }); \
        const size_t lds = F32Shape<K, NPC, A>::lds_bytes + (A == 2 ? (size_t)(g.BR < g.OH ? g.BR : g.OH) * 16 : 0);          \
        if (lds > 160 * 1024) return -1;                                                                                   \
        hipLaunchKernelGGL(kern, dim3((unsigned)nblocks), dim3(512), lds, s, (const float*)x, (const float*)w,             \
                           (const float*)add, (float*)y, g);                                                               \
    }
    const int mode = !add ? (K >= 13 && nblocks <= 256 && g.BR >= 12 ? -1 : 0) : g.OH == 2 * AH && g.OW == 2 * AW ? 1 : 2;
#define PDW_F32T_M(NPC) \
    if (mode == 0) PDW_F32T(NPC, 0) else if (mode == 1) PDW_F32T(NPC, 1) else if (mode == 2) PDW_F32T(NPC, 2) else PDW_F32T(NPC, (K >= 13 ? -1 : 0))
    if (npc == 16) {
        PDW_F32T_M(16)
    } else if (npc == 8) {
        PDW_F32T_M(8)
    } else {
        PDW_F32T_M(4)
    }
#undef PDW_F32T_M
#undef PDW_F32T
    return check_launch("dwconv_f32t");
}

// The forward convolutions of two problems (a block's scales, the second on the pooled input) in one grid, each in its own
// tiles and bands, as the separate launches would run them: where those leave compute units without work, the pair takes as
// long as the longer one (us: [2,32,32,32] and its half scale, filter 7, 7.1 + 5.8 -> 6.4; [3,57,61,100], filter 15, 17.6 +
// 10.7 -> 25.4; [32,56,56,64], filter 13, 39.9 + 16.0 -> 52.7).
struct F32Problem {
    const float *x, *w;
    float* y;
    F32Geom g;
    int npc, n;   // patches of a tile side by side; workgroups
};
struct F32Pair {
    F32Problem p[2];
};

template <int K>
__global__ __launch_bounds__(512, (f32t_waves<K, 0>())) void dwconv_f32t_pair_k(const F32Pair a) {
    const bool first = (int)blockIdx.x < a.p[0].n;
    const float *x = first ? a.p[0].x : a.p[1].x, *w = first ? a.p[0].w : a.p[1].w;
    float* const y = first ? a.p[0].y : a.p[1].y;
    const F32Geom g = first ? a.p[0].g : a.p[1].g;
    const int npc = first ? a.p[0].npc : a.p[1].npc, at = (int)blockIdx.x - (first ? 0 : a.p[0].n), n = first ? a.p[0].n : a.p[1].n;
    if (npc == 16) dwconv_f32_body<K, 16, 0>(x, w, nullptr, y, g, at, n);
    else if (npc == 8) dwconv_f32_body<K, 8, 0>(x, w, nullptr, y, g, at, n);
    else dwconv_f32_body<K, 4, 0>(x, w, nullptr, y, g, at, n);
}

// One problem of a launch of several, padding K / 2 (flip: the input gradient): its workgroups, and the LDS that it needs at least;
// false: not covered.
template <int K>
bool f32t_problem(F32Problem& p, long long& n, size_t& lds, const void* x, const void* w, void* y, int B, int H, int W, int C, bool flip) {
    if (!f32t_geom<K>(p.g, p.npc, n, B, H, W, C, K / 2, K / 2, flip)) return false;
    if (!f32t_pays<K>((long long)B * H * W * C, W, p.npc, false)) return false;
    for (const void* q : {x, w, (const void*)y})
        if (reinterpret_cast<uintptr_t>(q) & 15) return false;
    p.x = (const float*)x, p.w = (const float*)w, p.y = (float*)y, p.n = (int)n;
    const size_t need = p.npc == 16 ? F32Shape<K, 16>::lds_bytes : p.npc == 8 ? F32Shape<K, 8>::lds_bytes : F32Shape<K, 4>::lds_bytes;
    if (need > lds) lds = need;
    return true;
}

// -1: not covered (the caller makes two launches).  Padding K / 2.
template <int K>
int launch_f32t_pair(const void* x0, const void* w0, void* y0, int H0, int W0, const void* x1, const void* w1, void* y1, int H1,
                     int W1, int B, int C, hipStream_t s) {
    F32Pair a{};
    size_t lds = 0;
    long long n0, n1;
    if (!f32t_problem<K>(a.p[0], n0, lds, x0, w0, y0, B, H0, W0, C, false) || !f32t_problem<K>(a.p[1], n1, lds, x1, w1, y1, B, H1, W1, C, false))
        return -1;
    const long long total = n0 + n1;
    if (total > 0x7fffffffLL) return -1;
    static std::once_flag once;
    std::call_once(once, [] {
        (void)hipFuncSetAttribute((const void*)dwconv_f32t_pair_k<K>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    });
    hipLaunchKernelGGL(dwconv_f32t_pair_k<K>, dim3((unsigned)total), dim3(512), lds, s, a);
    return check_launch("dwconv_f32t_pair");
}

}  // namespace pdw
