// The products of dense_wide.hip in fp32 on the 16-bit matrix cores: an fp32 value is the sum of three bf16 values and a product of two
// the six products of parts that are not below its rounding (split_bf16.h), sixteen times the rate for six times the products.
//
// Tiles of BM x BN results by WM x WN wavefronts, stages of 32 inner values.  A stage is loaded into registers (16 bytes a lane,
// two stages ahead), split there, every value once for all the wavefronts that multiply it, and written as three planes of bf16 into
// one of two LDS buffers between the products of the other; one barrier a stage.  An operand stored [inner][result] is kept
// as it lies and read with ds_read_b64_tr_b16, as in dense_wide.hip.
//
// A value without such parts (infinite, NaN, or beyond 2^81) makes its workgroup's results again by plain multiply-adds, so that
// they are what fp32 arithmetic gives.  So does a result that is not finite: where x1 y1 overflows, x2 y1 may do so the other way, and
// an infinity would come out as NaN.  So do values that a lane holds of one stored row (TR: of four results) and that are all below
// 2^-100 and not all zero: the matrix cores take a bf16 value below 2^-126 as zero, which beside a value from 2^-100 on is at
// most 2^-26 of it and less than fp32's smallest normal value, and alone would be what the results consist of.
#pragma once
#include "common.h"
#include "dense_any_wgrad.h"
#include "split_bf16.h"
#include "tile_common.h"

namespace pdw {

namespace {

constexpr int kSplitBK = 32;   // inner values of a stage

// One operand of a tile: R results wide, staged by NT threads.  LDS planes: [result][32 inner], or (TR) [inner][R results], 16-byte
// pieces moved by the row so that a fragment read takes every bank once.
template <int R, bool TR, int NT>
struct SplitOperand {
    static constexpr int NL = R * 8 / NT;              // 16-byte loads per thread and stage
    static constexpr int PLANE = R * kSplitBK * 2;     // bytes
    static constexpr int CPR = TR ? R / 4 : 8;         // loads of a stored row
    static_assert(R * 8 % NT == 0, "whole loads");
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t off[NL];
    int kc[NL];      // first inner value of the piece (TR: its row)
    uint32_t step;   // bytes per stage

    static __device__ __forceinline__ int swz(int row, int c) {
        if constexpr (!TR) return c ^ ((row >> 2) & 3);
        else if constexpr (R == 128) return c ^ (4 * (row & 3));
        else return c ^ (4 * ((row >> 1) & 1));
    }
    // r0: first result; nres: results of the whole operand; inner values [kb, ke); ld: values of a stored row
    __device__ __forceinline__ void init(const float* p, int ld, long long r0, long long nres, long long kb, long long ke) {
        if constexpr (!TR) {
            const long long rows = nres - r0 < R ? nres - r0 : R;
            rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p + r0 * ld + kb), (short)0, (int)((rows - 1) * ld + (ke - kb)) * 4, 0x00020000);
            step = kSplitBK * 4;
        } else {
            rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p + kb * ld + r0), (short)0, (int)((ke - kb - 1) * ld + (nres - r0)) * 4, 0x00020000);
            step = (uint32_t)ld * kSplitBK * 4;
        }
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            const int slot = j * NT + (int)threadIdx.x, row = slot / CPR, c = slot % CPR;
            kc[j] = TR ? row : 4 * c;
            off[j] = r0 + (TR ? 4 * c : row) < nres ? (uint32_t)(row * ld + 4 * c) * 4u : kPast;
        }
    }
    __device__ __forceinline__ void request(split_f4 (&v)[NL], int st, int left) const {   // left: inner values from the stage's start
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            const uint32_t o = kc[j] < left ? off[j] + (uint32_t)st * step : kPast;
            v[j] = __builtin_bit_cast(split_f4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)o, 0, 0));
        }
    }
    static __device__ __forceinline__ void commit(char* buf, const split_f4 (&v)[NL], int j, float& seen, float (&top)[NL]) {
        top[j] = fmaxf(fmaxf(fabsf(v[j].x), fabsf(v[j].y)), fmaxf(fmaxf(fabsf(v[j].z), fabsf(v[j].w)), top[j]));
        const int slot = j * NT + (int)threadIdx.x, row = slot / CPR, c = slot % CPR;
        uint32_t lo[3], hi[3];
        split_pair(v[j].x, v[j].y, lo);
        split_pair(v[j].z, v[j].w, hi);
        seen = split_watch(hi, split_watch(lo, seen));
        char* const d = buf + row * (TR ? R * 2 : kSplitBK * 2) + swz(row, c >> 1) * 16 + (c & 1) * 8;
#pragma unroll
        for (int l = 0; l < 3; ++l) *reinterpret_cast<uint2*>(d + l * PLANE) = make_uint2(lo[l], hi[l]);
    }
    static __device__ __forceinline__ bool tiny(const float (&top)[NL]) {
        bool t = false;
#pragma unroll
        for (int j = 0; j < NL; ++j) t = t || (top[j] > 0.f && top[j] < 0x1p-100f);
        return t;
    }
    // eight inner values 16 kk + 8 (lane / 32) .. of result 32 t + lane % 32, of one part
    static __device__ __forceinline__ split_bf8 frag(const char* buf, int part, int t, int kk, int lane) {
        if constexpr (!TR) {
            const int row = 32 * t + (lane & 31), c = swz(row, 2 * kk + (lane >> 5));
            return *reinterpret_cast<const split_bf8*>(buf + part * PLANE + row * (kSplitBK * 2) + c * 16);
        } else {
            typedef short s4 __attribute__((ext_vector_type(4)));
            const int g = lane >> 4, i = lane & 15, col = 32 * t + 16 * (g & 1) + 4 * (i & 3);
            s4 h[2];
#pragma unroll
            for (int hh = 0; hh < 2; ++hh) {
                const int row = 16 * kk + 8 * (g >> 1) + 4 * hh + (i >> 2);
                h[hh] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (__attribute__((address_space(3))) s4*)(buf + part * PLANE + row * (R * 2) + swz(row, col >> 3) * 16 + (col & 7) * 2));
            }
            return __builtin_bit_cast(split_bf8, __builtin_shufflevector(h[0], h[1], 0, 1, 2, 3, 4, 5, 6, 7));
        }
    }
};

template <int BM, int BN, bool PART>
constexpr size_t split_lds() {
    constexpr size_t stages = (size_t)2 * 3 * (BM + BN) * kSplitBK * 2, out = PART ? 0 : (size_t)BM * (BN * 4 + 16);
    return stages > out ? stages : out;
}

// Results [M][N] = sum over k of a(m,k) b(n,k), as wide_gemm_body makes them.
template <int BM, int BN, int WM, int WN, bool TA, bool TB, bool PART, typename Args>
__device__ __forceinline__ void wide_split_body(const Args& g, int blk, int nblk) {
    constexpr int NT = 64 * WM * WN, FM = BM / 32 / WM, FN = BN / 32 / WN;
    typedef SplitOperand<BM, TA, NT> OpA;
    typedef SplitOperand<BN, TB, NT> OpB;
    constexpr int STAGE = 3 * (OpA::PLANE + OpB::PLANE), BOFF = 3 * OpA::PLANE;
    extern __shared__ __align__(16) char dsm[];
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave % WM, wn = wave / WM;
    int id = xcd_remap(blk, nblk);
    const int tn = id % g.nt;
    id /= g.nt;
    const int tm = id % g.mt, sp = id / g.mt;
    const long long m0 = (long long)tm * BM;
    const int n0 = tn * BN;
    const long long kb = sp * g.kper, ke = kb + g.kper < g.Kd ? kb + g.kper : g.Kd;
    OpA a;
    OpB b;
    a.init((const float*)g.a, g.lda, m0, g.M, kb, ke);
    b.init((const float*)g.b, g.ldb, n0, g.N, kb, ke);
    const int left = (int)(ke - kb), nst = (left + kSplitBK - 1) / kSplitBK;
    v16f acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    // (a sum over many rows in pieces of kSplitFlush stages, so that its error does not grow with a range's length)
    constexpr int kSplitFlush = 16;
    v16f total[PART ? FM : 1][PART ? FN : 1];
    if constexpr (PART) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) total[i][j] = acc[i][j];
    }
    float seen = 0.f, topa[OpA::NL] = {}, topb[OpB::NL] = {};
    split_f4 va[2][OpA::NL], vb[2][OpB::NL];
    auto request = [&](int p, int st) {
        a.request(va[p], st, left - st * kSplitBK);
        b.request(vb[p], st, left - st * kSplitBK);
    };
    constexpr int PIECES = OpA::NL + OpB::NL;
    auto commit = [&](int p, int piece, char* buf) {
        if (piece < OpA::NL) OpA::commit(buf, va[p], piece < OpA::NL ? piece : 0, seen, topa);
        else OpB::commit(buf + BOFF, vb[p], piece < OpA::NL ? 0 : piece - OpA::NL, seen, topb);
    };
    request(0, 0);
    request(1, 1);
#pragma unroll
    for (int e = 0; e < PIECES; ++e) commit(0, e, dsm);
    request(0, 2);
    // (the register buffers by name: stages in pairs, one past the last of zeros)
    for (int st = 0; st < nst; st += 2) {
        if constexpr (PART) {
            if (st % kSplitFlush == 0) {   // (uniform)
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j)
#pragma unroll
                        for (int r = 0; r < 16; ++r) total[i][j][r] += acc[i][j][r], acc[i][j][r] = 0.f;
            }
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const char* const cur = dsm + u * STAGE;
            char* const nxt = dsm + (u ^ 1) * STAGE;
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // this stage is in place, the other buffer read
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
                split_bf8 fa[FM][3], fb[FN][3];
#pragma unroll
                for (int l = 0; l < 3; ++l) {
#pragma unroll
                    for (int i = 0; i < FM; ++i) fa[i][l] = OpA::frag(cur, l, wm * FM + i, kk, lane);
#pragma unroll
                    for (int j = 0; j < FN; ++j) fb[j][l] = OpB::frag(cur + BOFF, l, wn * FN + j, kk, lane);
                }
                constexpr int of[6][2] = {{2, 0}, {1, 1}, {0, 2}, {1, 0}, {0, 1}, {0, 0}};   // parts: the small products first
#pragma unroll
                for (int n = 0; n < 6; ++n)
#pragma unroll
                    for (int i = 0; i < FM; ++i)
#pragma unroll
                        for (int j = 0; j < FN; ++j)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[j][of[n][0]], fa[i][of[n][1]], acc[i][j], 0, 0, 0);
#pragma unroll
                for (int e = kk * PIECES / 2; e < (kk + 1) * PIECES / 2; ++e) commit(u ^ 1, e, nxt);
            }
            request(u ^ 1, st + u + 3);
        }
    }
    auto out_of = [&](long long m, int n, float s) {   // (PART: the partial; else bias and the image's row are added)
        if constexpr (PART) {
            ((float*)g.y)[(size_t)sp * g.M * g.N + m * g.N + n] = s;
        } else {
            float add = 0.f;
            if (g.bias) add = ((const float*)g.bias)[n];
            if (g.rowbias) add += g.rowbias[(size_t)((uint32_t)m / (uint32_t)g.P) * g.N + n];
            ((float*)g.y)[m * g.N + n] = s + add;
        }
    };
    float finite = 0.f;   // (stays 0 while all results are)
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                if constexpr (PART) acc[i][j][r] += total[i][j][r];
                finite = fmaf(acc[i][j][r], 0.f, finite);
            }
    volatile uint32_t* const failed = reinterpret_cast<uint32_t*>(dsm);
    __syncthreads();
    if (tid == 0) *failed = 0;
    __syncthreads();
    if (split_failed(seen) || !(finite == 0.f) || OpA::tiny(topa) || OpB::tiny(topb)) *failed = 1;
    __syncthreads();
    if (*failed != 0) {   // (uniform)
        for (int r = tid; r < BM * BN; r += NT) {
            const long long m = m0 + r / BN;
            const int n = n0 + r % BN;
            if (m >= g.M || n >= g.N) continue;
            const float* const pa = (const float*)g.a + (TA ? kb * g.lda + m : m * g.lda + kb);
            const float* const pb = (const float*)g.b + (TB ? kb * g.ldb + n : (long long)n * g.ldb + kb);
            float s = 0.f;
            for (int k = 0; k < left; ++k) s = fmaf(pa[(long long)k * (TA ? g.lda : 1)], pb[(long long)k * (TB ? g.ldb : 1)], s);
            out_of(m, n, s);
        }
        return;
    }
    if constexpr (PART) {
        float* const out = (float*)g.y + (size_t)sp * g.M * g.N;
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            const long long m = m0 + (wm * FM + i) * 32 + l32;
            if (m >= g.M) continue;
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int n = n0 + (wn * FN + j) * 32 + 8 * q + 4 * h;
                    if (n < g.N)
                        *reinterpret_cast<float4*>(out + m * g.N + n) =
                            make_float4(acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
                }
        }
    } else {
        // bias and per-image row, then through LDS so that the stores are whole 16-byte pieces in order
        constexpr int TP = BN + 4, CPR = BN / 4;
        float* const tile = reinterpret_cast<float*>(dsm);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            const int mr = (wm * FM + i) * 32 + l32;
            const long long m = m0 + mr < g.M ? m0 + mr : g.M - 1;
            const float* const rb = g.rowbias ? g.rowbias + (size_t)((uint32_t)m / (uint32_t)g.P) * g.N : nullptr;
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int nr = (wn * FN + j) * 32 + 8 * q + 4 * h, n = n0 + nr < g.N ? n0 + nr : 0;
                    float4 add = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (g.bias) add = *reinterpret_cast<const float4*>((const float*)g.bias + n);
                    if (rb) {
                        const float4 t = *reinterpret_cast<const float4*>(rb + n);
                        add.x += t.x, add.y += t.y, add.z += t.z, add.w += t.w;
                    }
                    *reinterpret_cast<float4*>(tile + mr * TP + nr) = make_float4(acc[i][j][4 * q] + add.x, acc[i][j][4 * q + 1] + add.y,
                                                                                  acc[i][j][4 * q + 2] + add.z, acc[i][j][4 * q + 3] + add.w);
                }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < BM * CPR / NT; ++j) {
            const int s = j * NT + tid, row = s / CPR, c = s % CPR;
            if (m0 + row < g.M && n0 + c * 4 < g.N)
                *reinterpret_cast<uint4*>((float*)g.y + (m0 + row) * g.N + n0 + c * 4) = *reinterpret_cast<const uint4*>(tile + row * TP + c * 4);
        }
    }
}

}  // namespace

}  // namespace pdw
