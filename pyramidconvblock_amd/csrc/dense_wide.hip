// Dense layers of wide blocks (16-bit types, widths that are multiples of 8) and of fp32 blocks (multiples of 4): all three
// products of an nn.Linear on tiles of 128 x 128 (or 64) results, the products of conv_block.py:37, 44 for any dim.
//
//   rows:   Y[n,o]  = sum_k X[n,k] W(o,k) + bias[o] + rowbias[n / P][o]     (W stored [o][k], or [k][o] for the input gradient)
//   wgrad:  dW[m,o] = sum_n A[n,m] B[n,o]                                    (fp32 partials over row ranges)
//
// What bounds it: the matrix pipe from a width of about 600 on, HBM below.  A stage is 128 bytes of the inner dimension
// (64 values, in fp32 32) of both operands, moved by the direct global-to-LDS loads (16 bytes a lane, no registers in between) into one of two
// buffers while the other is multiplied; one barrier a stage.  Where a launch leaves compute units with one workgroup each there are
// four such buffers, since nothing else covers a stage's trip to memory.  Operands whose inner dimension is not the contiguous one
// (both of the weight gradient, the weight of the input gradient) are staged as they lie and read with
// ds_read_b64_tr_b16, which hands every lane four values down a column, so there is no transposing pass over memory and
// no byte shuffling.  The 16-byte pieces of a staged row are permuted by the row (the loads' lanes choose the global piece,
// since their LDS side is fixed to lane order), so that the fragment reads of both kinds fall on all 64 banks once.
// Measured (bf16, us; in brackets the library product it replaces): [16384,1152] -> 576 27 (34), its input gradient 30
// (48), its weight gradient 32 + its share of the summation (a batched product over 128 slabs and their sum: 160 + 150).
// fp32 (v_mfma_f32_32x32x2_f32, a sixteenth of the rate, so that the LDS and its reads down a column value by value are no
// matter), us, dense_any.hip -> here: [100352,128] -> 64 28.7 -> 22.8, its input gradient 32.3 -> 25.6 (77 MB, 10.5 us of matrix
// pipe); [10431,200] -> 100 16.0 -> 11.4; [20000,256] -> 128 26.5 -> 18.7; [2048,64] -> 32 5.1 -> 3.8.
// Out-of-range rows, columns and the inner tail read as zero through the buffer descriptors; nothing is branched around.
#include <stdint.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "common.h"
#include "dense_any_wgrad.h"
#include "kernels.h"
#include "mean_any.h"
#include "reduce_parts.h"
#include "tile_common.h"

namespace pdw {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef short v4s __attribute__((ext_vector_type(4)));
typedef short v8s __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) char lds_char;

constexpr int kRowBytes = 128;              // inner bytes per stage: 64 values of 16 bits, 32 of fp32
template <typename T>
constexpr int kBK = kRowBytes / (int)sizeof(T);

__device__ __forceinline__ v16f mfma(v8s a, v8s b, v16f c, bf16_t) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
}
__device__ __forceinline__ v16f mfma(v8s a, v8s b, v16f c, f16_t) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
}
// (a lane's four values are inner values 8 kk + 4 (lane / 32) + t, of both operands: the order of a sum's terms)
__device__ __forceinline__ v16f mfma(v8s a, v8s b, v16f c, float) {
    const v4f x = __builtin_bit_cast(v4f, a), y = __builtin_bit_cast(v4f, b);
    const float x0 = x.x, x1 = x.y, x2 = x.z, x3 = x.w, y0 = y.x, y1 = y.y, y2 = y.z, y3 = y.w;
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(x0, y0, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(x1, y1, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(x2, y2, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x2f32(x3, y3, c, 0, 0, 0);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}

// Rows of a tensor [images][2 h][2 w][] taken by quads, the 2 x 2 pixels of one pooled pixel: row 4 q + 2 dy + dx is pixel (2 y + dy, 2 x + dx)
// of pooled pixel q, so that a tile of rows holds whole quads whatever the extents are.  (Images are stacked: H = 2 h.)
struct QuadArgs {
    void* pool;       // [images][h][w][]: the mean of each quad's results
    int w;
    uint32_t magic;   // 2^32 / w rounded up (w > 1): x / w for x w < 2^32
};
struct QuadRows {
    uint32_t pix0, x0;   // first pixel of the row pair of the tile's first quad, and that quad's place in it
    int w;
    uint32_t magic;
    __device__ __forceinline__ void init(const QuadArgs& g, long long quad0) {
        const uint32_t pair = (uint32_t)quad0 / (uint32_t)g.w;
        w = g.w, magic = g.magic, x0 = (uint32_t)quad0 - pair * (uint32_t)w, pix0 = 4 * pair * (uint32_t)w;
    }
    __device__ __forceinline__ uint32_t pixel(int row) const {   // of the tile's row, from pix0
        const uint32_t t = x0 + (uint32_t)(row >> 2), dy = w == 1 ? t : __umulhi(t, magic), x = t - dy * (uint32_t)w;
        return (2 * dy + (uint32_t)(row >> 1 & 1)) * 2 * (uint32_t)w + 2 * x + (uint32_t)(row & 1);
    }
};

// One operand of a tile: R results wide, kBK inner values per stage, staged by the workgroup's 256 threads.
// TR = false: stored [result][inner] (pitch ld): LDS rows of 128 bytes, 8 pieces each, piece c of row r at c ^ (r / 2 % 8).
// TR = true: stored [inner][result]: LDS rows of R values; pieces moved in groups (64 bytes; fp32 128) by the row, so that the
// rows that a read takes together (the four of a transposing read; in fp32 two, four apart) lie on different banks.
template <typename T, int R, bool TR>
struct Operand {
    static constexpr int ES = (int)sizeof(T), VE = 16 / ES;
    static constexpr int NL = R * kRowBytes / 16 / 256;   // loads per thread and stage
    static constexpr int CPR = TR ? R / VE : 8;           // pieces per LDS row
    static constexpr int BYTES = R * kRowBytes;
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t off[NL];
    int kc[NL];          // first inner value of the piece (TR: its row)
    uint32_t step;       // bytes per stage

    static __device__ __forceinline__ int swz(int row, int c) {
        if constexpr (!TR) return c ^ ((row >> 1) & 7);
        else if constexpr (ES == 4) return c ^ (8 * ((row >> 2) & 1));
        else if constexpr (R == 128) return c ^ (4 * (row & 3));
        else return c ^ (4 * ((row >> 1) & 1));
    }
    // r0: first result; nres: results of the whole operand; inner values [kb, ke)
    __device__ __forceinline__ void init(const char* p, int ld, long long r0, long long nres, long long kb, long long ke) {
        const int tid = threadIdx.x;
        if constexpr (!TR) {
            const long long rows = nres - r0 < R ? nres - r0 : R;
            rsrc = rsrc_of(p + (r0 * ld + kb) * ES, (uint32_t)((rows - 1) * ld + (ke - kb)) * ES);
            step = kRowBytes;
        } else {
            rsrc = rsrc_of(p + (kb * ld + r0) * ES, (uint32_t)((ke - kb - 1) * ld + (nres - r0)) * ES);
            step = (uint32_t)ld * kRowBytes;
        }
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            const int slot = j * 256 + tid, row = slot / CPR, c = swz(row, slot % CPR);
            if constexpr (!TR) {
                kc[j] = c * VE;
                off[j] = r0 + row < nres ? (uint32_t)(row * ld + c * VE) * ES : kPast;
            } else {
                kc[j] = row;
                off[j] = r0 + c * VE < nres ? (uint32_t)(row * ld + c * VE) * ES : kPast;
            }
        }
    }
    // results of a tensor that leaves some out (RowMap): result c at its row c % seg + val (c / seg), zero where c % seg >= val
    __device__ __forceinline__ void init(const char* p, int ld, long long r0, long long nres, long long kb, long long ke, const RowMap& map) {
        static_assert(!TR, "stored by results");
        rsrc = rsrc_of(p + kb * ES, (uint32_t)((2 * map.val - 1) * ld + (ke - kb)) * ES);
        step = kRowBytes;
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            const int slot = j * 256 + (int)threadIdx.x, row = slot / CPR, c = swz(row, slot % CPR);
            const int res = (int)r0 + row, hi = res >= map.seg, r = res - hi * map.seg;
            kc[j] = c * VE;
            off[j] = r < map.val && res < nres ? (uint32_t)((r + hi * map.val) * ld + c * VE) * ES : kPast;
        }
    }
    // rows by quads from `quad0` on, of `quads`
    __device__ __forceinline__ void init(const char* p, int ld, const QuadRows& rows, long long quad0, long long quads) {
        static_assert(!TR, "stored by results");
        const long long bytes = (4 * quads - rows.pix0) * ld * ES;
        rsrc = rsrc_of(p + (long long)rows.pix0 * ld * ES, (uint32_t)(bytes < 0x7fffffffLL ? bytes : 0x7fffffffLL));
        step = kRowBytes;
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            const int slot = j * 256 + (int)threadIdx.x, row = slot / CPR, c = swz(row, slot % CPR);
            kc[j] = c * VE;
            off[j] = quad0 + (row >> 2) < quads ? (rows.pixel(row) * (uint32_t)ld + (uint32_t)(c * VE)) * ES : kPast;
        }
    }
    // requests stage `st` (inner values left from its start: left) into buf
    __device__ __forceinline__ void request(lds_char* buf, int st, int left) const {
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            const uint32_t o = kc[j] < left ? off[j] + (uint32_t)st * step : kPast;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(buf + (j * 256 + wave * 64) * 16),
                                                     16, (int)o, 0, 0, 0);
        }
    }
    // this lane's 16 bytes of inner values (2 VE kk + VE (lane / 32) ..) of result 32 t + lane % 32
    static __device__ __forceinline__ v8s frag(const lds_char* buf, int t, int kk, int lane) {
        if constexpr (!TR) {
            const int row = 32 * t + (lane & 31), c = swz(row, 2 * kk + (lane >> 5));
            return *(const __attribute__((address_space(3))) v8s*)(buf + row * kRowBytes + c * 16);
        } else if constexpr (ES == 4) {
            const int col = 32 * t + (lane & 31), row = 8 * kk + 4 * (lane >> 5);
            const lds_char* const p = buf + row * (R * 4) + swz(row, col >> 2) * 16 + (col & 3) * 4;
            float e[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) e[i] = *(const __attribute__((address_space(3))) float*)(p + i * (R * 4));
            const v4f v = {e[0], e[1], e[2], e[3]};
            return __builtin_bit_cast(v8s, v);
        } else {
            const int g = lane >> 4, i = lane & 15;
            const int col = 32 * t + 16 * (g & 1) + 4 * (i & 3);
            v4s h[2];
#pragma unroll
            for (int hh = 0; hh < 2; ++hh) {
                const int row = 16 * kk + 8 * (g >> 1) + 4 * hh + (i >> 2);
                h[hh] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (__attribute__((address_space(3))) v4s*)(buf + row * (R * 2) + swz(row, col >> 3) * 16 + (col & 7) * 2));
            }
            return __builtin_shufflevector(h[0], h[1], 0, 1, 2, 3, 4, 5, 6, 7);
        }
    }
};

// Fragments read by hand, for the loop that keeps requests in flight across LDS reads (the compiler would let each such read wait
// for all of them: it cannot tell the stages apart); the waits are that loop's own.
template <typename T, int R, bool TR>
struct HandFragments {
    typedef Operand<T, R, TR> Op;
    static_assert(sizeof(T) == 2, "16-bit values");
    static constexpr int READS = TR ? 2 : 1;   // LDS instructions of a fragment
    // per lane and in a stage, but for constants: (TR) where fragment t's values of kk = 0 lie, else those of kk = n and t = 0
    static __device__ __forceinline__ uint32_t at(int n, int lane) {
        if constexpr (!TR) {
            const int row = lane & 31;
            return (uint32_t)(row * kRowBytes + Op::swz(row, 2 * n + (lane >> 5)) * 16);
        } else {
            const int g = lane >> 4, i = lane & 15, col = 32 * n + 16 * (g & 1) + 4 * (i & 3), row = 8 * (g >> 1) + (i >> 2);
            return (uint32_t)(row * (R * 2) + Op::swz(row, col >> 3) * 16 + (col & 7) * 2);
        }
    }
    template <int TILE, int KK>
    static __device__ __forceinline__ v8s read(uint32_t p) {   // p: stage + at
        if constexpr (!TR) {
            v8s f;
            asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(f) : "v"(p), "n"(TILE * 32 * kRowBytes));
            return f;
        } else {
            v4s h0, h1;
            asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(h0) : "v"(p), "n"(16 * KK * R * 2));
            asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(h1) : "v"(p), "n"((16 * KK + 4) * R * 2));
            return __builtin_shufflevector(h0, h1, 0, 1, 2, 3, 4, 5, 6, 7);
        }
    }
};

// Until all but the newest N LDS instructions are done, from when on what the others read may be used.
template <int N, int FM, int FN>
__device__ __forceinline__ void wait_fragments(v8s (&a)[FM], v8s (&b)[FN]) {
    asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N < 15 ? N : 15));
#pragma unroll
    for (int i = 0; i < FM; ++i) asm volatile("" : "+v"(a[i]));
#pragma unroll
    for (int j = 0; j < FN; ++j) asm volatile("" : "+v"(b[j]));
    __builtin_amdgcn_sched_barrier(0);
}

template <int N, int I = 0, typename F>
__device__ __forceinline__ void for_each(F f) {   // f(0) .. f(N - 1), the index a constant
    if constexpr (I < N) f(std::integral_constant<int, I>()), for_each<N, I + 1>(f);
}

struct WideArgs {
    const void *a, *b, *bias;
    const float* rowbias;
    void* y;              // T, or the fp32 partials
    long long M, Kd;      // results along a; inner extent
    int N, lda, ldb, P;   // results along b
    int mt, nt, splits;
    long long kper;       // inner values per split (a multiple of 64)
    RowMap map;           // of b's results (16-bit rows, stored by results)
};

// Results [M][N] = sum over k of a(m,k) b(n,k).  The b operand is the matrix instruction's first, so that a lane holds
// four consecutive n of one m.  Wavefronts 2 x 2 over the tile.
// Workgroups of a compute unit: fp32 has registers and LDS for more than two of the smaller tiles.
template <typename T, int BM, int BN>
constexpr int kWideOccupancy = sizeof(T) == 4 ? (BM * BN <= 64 * 64 ? 4 : BM * BN <= 128 * 64 ? 3 : 2) : 2;

// QUAD: a's rows by quads (M of them), and the mean of each quad's results as they are stored.
template <typename T, int BM, int BN, bool TA, bool TB, bool PART, int STAGES = 2, bool MAP = false, bool QUAD = false>
__device__ __forceinline__ void wide_gemm_body(const WideArgs& g, int blk, int nblk, const QuadArgs& qa = QuadArgs{}) {
    typedef Operand<T, BM, TA> OpA;
    typedef Operand<T, BN, TB> OpB;
    constexpr int BK = kBK<T>, KK = 4;          // inner values of a stage; fragments of it
    constexpr int STAGE = OpA::BYTES + OpB::BYTES;
    constexpr int FM = BM / 64, FN = BN / 64;   // 32-result fragments per wavefront
    extern __shared__ __align__(16) char dsm[];
    lds_char* const sm = (lds_char*)dsm;
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave & 1, wn = wave >> 1;
    // tiles of one row range next to each other on one XCD: they read the same rows
    int id = xcd_remap(blk, nblk);
    const int tn = id % g.nt;
    id /= g.nt;
    const int tm = id % g.mt, sp = id / g.mt;
    const long long m0 = (long long)tm * BM;
    const int n0 = tn * BN;
    const long long kb = sp * g.kper, ke = kb + g.kper < g.Kd ? kb + g.kper : g.Kd;
    OpA a;
    OpB b;
    QuadRows quad;
    if constexpr (QUAD) {
        quad.init(qa, m0 / 4);
        a.init((const char*)g.a, g.lda, quad, m0 / 4, g.M / 4);
    } else {
        a.init((const char*)g.a, g.lda, m0, g.M, kb, ke);
    }
    // (a kernel of its own for a RowMap: chosen inside one, the two cost other layers up to 0.6 us of 10)
    if constexpr (MAP) b.init((const char*)g.b, g.ldb, n0, g.N, kb, ke, g.map);
    else b.init((const char*)g.b, g.ldb, n0, g.N, kb, ke);
    const int left = (int)(ke - kb), nst = (left + BK - 1) / BK;
    v16f acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    if constexpr (STAGES == 2) {
        a.request(sm, 0, left);
        b.request(sm + OpA::BYTES, 0, left);
        for (int st = 0; st < nst; ++st) {
            lds_char* const cur = sm + (st & 1) * STAGE;
            lds_char* const nxt = sm + ((st & 1) ^ 1) * STAGE;
            // this stage has arrived, and every wavefront is done with the buffer that the next one goes to
            asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
            // all fragments of the stage first, then the next stage's requests, then the products: an LDS read behind a
            // request in program order would wait for it (the compiler cannot tell the two buffers apart)
            v8s fa[KK][FM], fb[KK][FN];
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) {
#pragma unroll
                for (int i = 0; i < FM; ++i) fa[kk][i] = OpA::frag(cur, wm * FM + i, kk, lane);
#pragma unroll
                for (int j = 0; j < FN; ++j) fb[kk][j] = OpB::frag(cur + OpA::BYTES, wn * FN + j, kk, lane);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (st + 1 < nst) {
                a.request(nxt, st + 1, left - (st + 1) * BK);
                b.request(nxt + OpA::BYTES, st + 1, left - (st + 1) * BK);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int kk = 0; kk < KK; ++kk)
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j) acc[i][j] = mfma(fb[kk][j], fa[kk][i], acc[i][j], T());
        }
    } else {
        // STAGES in LDS and all but two of them on their way: a launch that leaves compute units with one workgroup each has
        // nothing else to cover a trip to memory with.  Fragments are read one product ahead, across the stages too.
        typedef HandFragments<T, BM, TA> HA;
        typedef HandFragments<T, BN, TB> HB;
        constexpr int LOADS = OpA::NL + OpB::NL, READS = FM * HA::READS + FN * HB::READS, NA = TA ? FM : KK, NB = TB ? FN : KK;
        static_assert(STAGES > 2 && (STAGES - 2) * LOADS < 64, "requests in flight");
        const uint32_t lds0 = (uint32_t)(uintptr_t)sm;
        uint32_t ata[NA], atb[NB];
#pragma unroll
        for (int n = 0; n < NA; ++n) ata[n] = lds0 + (TA ? HA::at(wm * FM + n, lane) : HA::at(n, lane) + (uint32_t)(wm * FM * 32 * kRowBytes));
#pragma unroll
        for (int n = 0; n < NB; ++n)
            atb[n] = lds0 + OpA::BYTES + (TB ? HB::at(wn * FN + n, lane) : HB::at(n, lane) + (uint32_t)(wn * FN * 32 * kRowBytes));
        auto request = [&](int st, int slot) {   // (past the last stage: zeros, so that every stage has its requests)
            a.request(sm + slot * STAGE, st, left - st * BK);
            b.request(sm + slot * STAGE + OpA::BYTES, st, left - st * BK);
        };
        v8s fa[2][FM], fb[2][FN];
        auto fragments = [&](int slot, auto kk) {
            const uint32_t buf = (uint32_t)(slot * STAGE);
            for_each<FM>([&](auto i) { fa[kk & 1][i] = HA::template read<TA ? 0 : i, kk>(buf + ata[TA ? i : kk]); });
            for_each<FN>([&](auto j) { fb[kk & 1][j] = HB::template read<TB ? 0 : j, kk>(buf + atb[TB ? j : kk]); });
            __builtin_amdgcn_sched_barrier(0);
        };
        constexpr std::integral_constant<int, 0> first;
#pragma unroll
        for (int st = 0; st < STAGES - 1; ++st) request(st, st);
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((STAGES - 2) * LOADS) : "memory");
        fragments(0, first);
        int slot = 0;
        for (int st = 0; st < nst; ++st) {
            const int next = slot + 1 == STAGES ? 0 : slot + 1, before = slot == 0 ? STAGES - 1 : slot - 1;
            for_each<KK>([&](auto kk) {
                if constexpr (kk + 1 < KK) {
                    fragments(slot, std::integral_constant<int, kk + 1>());
                } else {
                    // the next stage has arrived, and every wavefront is done with the one before this, whose place is requested into
                    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((STAGES - 3) * LOADS) : "memory");
                    fragments(next, first);
                    request(st + STAGES - 1, before);
                }
                wait_fragments<READS>(fa[kk & 1], fb[kk & 1]);
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j) acc[i][j] = mfma(fb[kk & 1][j], fa[kk & 1][i], acc[i][j], T());
                __builtin_amdgcn_sched_barrier(0);
            });
            slot = next;
        }
        // (the last turn has read fragments that nothing uses: their registers are given away only behind this wait)
        wait_fragments<0>(fa[0], fb[0]);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    if constexpr (PART && sizeof(T) == 4) {   // (tiles of 64, four to a compute unit: nothing to win by the other way)
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
    } else if constexpr (PART) {
        // through LDS: as they lie in registers a store would write 16 bytes of each of 32 rows ([3136,768]^T [3136,384] 18.6 -> 17.5 us)
        constexpr int TP = BN + 4, CPR = BN / 4;
        __syncthreads();
        float* const tile = reinterpret_cast<float*>(dsm);
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<float4*>(tile + ((wm * FM + i) * 32 + l32) * TP + (wn * FN + j) * 32 + 8 * q + 4 * h) =
                        make_float4(acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
        __syncthreads();
        float* const out = (float*)g.y + (size_t)sp * g.M * g.N;
#pragma unroll
        for (int j = 0; j < BM * CPR / 256; ++j) {
            const int s = j * 256 + tid, row = s / CPR, c = s % CPR;
            if (m0 + row < g.M && n0 + c * 4 < g.N)
                *reinterpret_cast<float4*>(out + (m0 + row) * g.N + n0 + c * 4) = *reinterpret_cast<const float4*>(tile + row * TP + c * 4);
        }
    } else {
        // bias and per-image row in fp32, then through LDS so that the stores are whole 16-byte pieces in order
        constexpr int VE = 16 / (int)sizeof(T), TP = BN + VE;
        __syncthreads();
        T* const tile = reinterpret_cast<T*>(dsm);
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
                    float v[4] = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
                    float add[4] = {0.f, 0.f, 0.f, 0.f};
                    if (g.bias) load_f32<T, 4>((const T*)g.bias + n, add);
                    if (rb) {
                        const float4 t = *reinterpret_cast<const float4*>(rb + n);
                        add[0] += t.x, add[1] += t.y, add[2] += t.z, add[3] += t.w;
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] += add[e];
                    store_f32<T, 4>(tile + mr * TP + nr, v);
                }
        }
        __syncthreads();
        constexpr int CPR = BN / VE;
        if constexpr (QUAD) {   // a quad's pieces by one thread, and their mean in avgpool_fwd_item's order
#pragma unroll
            for (int s = tid; s < BM / 4 * CPR; s += 256) {
                const int row = s / CPR * 4, c = s % CPR;
                if (m0 + row >= g.M || n0 + c * VE >= g.N) continue;
                T* const y = (T*)g.y + (quad.pix0 + (long long)quad.pixel(row)) * g.N + n0 + c * VE;
                ChanVec<T, VE> v[4];
                float o[VE];
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = *reinterpret_cast<const ChanVec<T, VE>*>(tile + (row + r) * TP + c * VE);
#pragma unroll
                for (int r = 0; r < 4; ++r) *reinterpret_cast<ChanVec<T, VE>*>(y + (long long)((r >> 1) * 2 * quad.w + (r & 1)) * g.N) = v[r];
#pragma unroll
                for (int e = 0; e < VE; ++e) o[e] = (((to_f32(v[0].v[e]) + to_f32(v[1].v[e])) + to_f32(v[2].v[e])) + to_f32(v[3].v[e])) * 0.25f;
                store_f32<T, VE>((T*)qa.pool + ((m0 + row) / 4) * g.N + n0 + c * VE, o);
            }
        } else {
#pragma unroll
            for (int j = 0; j < BM * CPR / 256; ++j) {
                const int s = j * 256 + tid, row = s / CPR, c = s % CPR;
                if (m0 + row < g.M && n0 + c * VE < g.N)
                    *reinterpret_cast<uint4*>((T*)g.y + (m0 + row) * g.N + n0 + c * VE) = *reinterpret_cast<const uint4*>(tile + row * TP + c * VE);
            }
        }
    }
}

template <typename T, int BM, int BN, bool TA, bool TB, bool PART, int STAGES, bool MAP = false>
__global__ __launch_bounds__(256, (STAGES == 2 ? kWideOccupancy<T, BM, BN> : 1)) void wide_gemm_k(WideArgs g) {
    wide_gemm_body<T, BM, BN, TA, TB, PART, STAGES, MAP>(g, blockIdx.x, gridDim.x);
}

// The first layer of a block whose pooled extents are exact halves: the pool of its result in the product's store, where it lies in LDS
// anyway (its rows go by quads for that), and the column sums of its input (mean_any.h) by workgroups of their own behind the
// product's.  Instead of a launch that reads both again and of its start-up: what bounds it is the product (matrix pipe or HBM), the pool and
// the rows' order cost 2 us of 30, the sums 1 to 4.  us, the product and that launch -> this: [100352,128] -> 64 fp32 23.6 + 13.0 -> 28.7;
// [25600,400] -> 200 fp32 53.1 + 12.9 -> 53.3; [16384,1152] -> 576 fp16 29.4 + 11.5 -> 30.8; [100352,256] -> 128 bf16 20.4 + 14.2 -> 25.2;
// [3200,640] -> 320 8.3 + 4.0 -> 9.4; [2048,64] -> 32 fp32 4.5 + 2.9 -> 5.4.  Where the pool needs a launch of its own (odd extents) the sums stay
// there: [10431,200] -> 100 fp32 11.2 + 6.1, riding here 12.2 + 5.4; [1500,920] -> 464 bf16 10.4 + 5.2 and 14.7 + 5.1 (two stages, not four).
template <typename T, int BM, int BN, int STAGES>
__global__ __launch_bounds__(256, (STAGES == 2 ? kWideOccupancy<T, BM, BN> : 1)) void wide_first_k(WideArgs g, QuadArgs qa, ColsumJob sums, int nrows) {
    extern __shared__ __align__(16) char dsm[];
    const int blk = blockIdx.x;
    if (blk < nrows) wide_gemm_body<T, BM, BN, false, false, false, STAGES, false, true>(g, blk, nrows, qa);
    else colsum_body<T, true>(sums, blk - nrows, (float*)dsm);
}

// With the weights by a RowMap, and their packing (pack_weights.h) last.
template <typename T, int BM, int BN, int STAGES>
__global__ __launch_bounds__(256, (STAGES == 2 ? kWideOccupancy<T, BM, BN> : 1)) void wide_first_pack_k(WideArgs g, QuadArgs qa, ColsumJob sums, int nrows,
                                                                                                     int nsums, PackArgs pack) {
    extern __shared__ __align__(16) char dsm[];
    const int blk = blockIdx.x;
    if (blk < nrows) wide_gemm_body<T, BM, BN, false, false, false, STAGES, true, true>(g, blk, nrows, qa);
    else if (blk < nrows + nsums) colsum_body<T, true>(sums, blk - nrows, (float*)dsm);
    else pack_weights_body(pack, blk - nrows - nsums);
}

// Both products that read the gradient of a layer's output, as one launch: the weight gradient's nw workgroups (tiles of WM x WN
// of this file; WM = 0: the kernel without LDS, dense_any_wgrad.h), which are the longer ones, then the input gradient's.  A
// launch of its own leaves part of the chip idle in its last round and pays the ramp; together they are dealt as one.
// us, two launches -> one: [100352,128] <- 64 fp32 44.7 -> 41.0, 64 <- 128 48.4 -> 43.0 (153 and 180 MB); [10431,200] <- 104 bf16 13.4
// -> 8.8; [16384,1152] <- 576 fp16 66.5 -> 61.4, 576 <- 1152 71.7 -> 68.1; [2048,64] <- 32 fp32 8.6 -> 4.9.
template <typename T, int BM, int BN, int WM, int WN, int STAGES>
__global__ __launch_bounds__(256, (STAGES == 2 ? kWideOccupancy<T, BM, BN> : 1)) void wide_pair_k(WideArgs rows, WideArgs wgrad, AnyWgradArgs any, int nw) {
    const int blk = blockIdx.x;
    if (blk >= nw) {
        wide_gemm_body<T, BM, BN, false, true, false, STAGES>(rows, blk - nw, gridDim.x - nw);
    } else if constexpr (WM != 0) {
        wide_gemm_body<T, WM, WN, true, true, true, STAGES>(wgrad, blk, nw);
    } else {
        const int group = blk / any.chunks;
        dense_any_wgrad_body<T>(any, blk - group * any.chunks, group);
    }
}

// And with the column sums of the gradient (mean_any.h) behind them.
template <typename T, int BM, int BN, int WM, int WN, int STAGES>
__global__ __launch_bounds__(256, (STAGES == 2 ? kWideOccupancy<T, BM, BN> : 1)) void wide_pair_sums_k(WideArgs rows, WideArgs wgrad, AnyWgradArgs any, int nw,
                                                                                                    ColsumJob sums, int nrows) {
    extern __shared__ __align__(16) char dsm[];
    const int blk = blockIdx.x;
    if (blk >= nw + nrows) {
        colsum_body<T, true>(sums, blk - nw - nrows, (float*)dsm);
    } else if (blk >= nw) {
        wide_gemm_body<T, BM, BN, false, true, false, STAGES>(rows, blk - nw, nrows);
    } else if constexpr (WM != 0) {
        wide_gemm_body<T, WM, WN, true, true, true, STAGES>(wgrad, blk, nw);
    } else {
        const int group = blk / any.chunks;
        dense_any_wgrad_body<T>(any, blk - group * any.chunks, group);
    }
}

template <typename T, int BM, int BN, bool PART, int STAGES>
constexpr size_t wide_lds() {
    constexpr size_t stages = (size_t)STAGES * (BM + BN) * kRowBytes, out = (size_t)BM * (BN * (PART ? 4 : sizeof(T)) + 16);
    return stages > out ? stages : out;
}

// Launches that kDeep stages in LDS are for: 16-bit ones whose workgroups are all on the chip at once with them, and whose sums have
// `least` stages or more (us, two stages -> four: [2128,920] -> 464, 136 workgroups of 15 stages, 12.0 -> 9.65, [1568,1024] -> 512 11.8 -> 9.2,
// [3136,768] -> 384 10.1 -> 8.2; of five stages or fewer the same or up to 0.4 more.  fp32's products take
// longer than a stage's trip: [10431,200] -> 100 11.7 -> 12.5, [12544,256] -> 128 12.7 -> 13.2, [2048,96] -> 48 4.6 -> 4.9).
constexpr int kDeep = 4;
template <typename T>
constexpr bool goes_deep(long long n, size_t lds, long long inner, int least) {
    return sizeof(T) == 2 && inner >= least * kBK<T> && n <= 256LL * (long long)(160 * 1024 / lds);
}

template <typename T, int BM, int BN, int WM, int WN, int STAGES>
int pair_go(const WideArgs& rows, const WideArgs& wgrad, const AnyWgradArgs& any, int nw, const ColsumJob* sums, hipStream_t s) {
    constexpr size_t a = wide_lds<T, BM, BN, false, STAGES>(), b = WM != 0 ? wide_lds<T, WM, WN, true, STAGES>() : 0, lds = a > b ? a : b;
    const long long nrows = (long long)rows.mt * rows.nt, n = nw + nrows + (sums ? colsum_workgroups(*sums) : 0);
    if (n > 0x7fffffffLL) return -1;
    if constexpr (STAGES == kDeep) {
        if (!goes_deep<T>(n, lds, rows.Kd, 4)) return pair_go<T, BM, BN, WM, WN, 2>(rows, wgrad, any, nw, sums, s);
    }
    if constexpr (lds > 64 * 1024) {
        static std::once_flag once;
        std::call_once(once, [] {
            for (const void* k : {(const void*)wide_pair_k<T, BM, BN, WM, WN, STAGES>, (const void*)wide_pair_sums_k<T, BM, BN, WM, WN, STAGES>})
                (void)hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        });
    }
    if (sums) {
        hipLaunchKernelGGL((wide_pair_sums_k<T, BM, BN, WM, WN, STAGES>), dim3((unsigned)n), dim3(256), lds, s, rows, wgrad, any, nw, *sums, (int)nrows);
        return check_launch("wide_pair_sums");
    }
    hipLaunchKernelGGL((wide_pair_k<T, BM, BN, WM, WN, STAGES>), dim3((unsigned)n), dim3(256), lds, s, rows, wgrad, any, nw);
    return check_launch("wide_pair");
}

template <typename T, int BM, int BN, bool TA, bool TB, bool PART, int STAGES = kDeep, bool MAP = false>
int wide_go(const WideArgs& g, hipStream_t s) {
    constexpr size_t lds = wide_lds<T, BM, BN, PART, STAGES>();
    if constexpr (STAGES == kDeep) {
        if (!goes_deep<T>((long long)g.mt * g.nt * g.splits, lds, PART ? g.kper : g.Kd, PART ? 3 : 6)) return wide_go<T, BM, BN, TA, TB, PART, 2, MAP>(g, s);
    }
    if constexpr (lds > 64 * 1024) {
        static std::once_flag once;
        std::call_once(once, [] {
            (void)hipFuncSetAttribute((const void*)wide_gemm_k<T, BM, BN, TA, TB, PART, STAGES, MAP>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        });
    }
    hipLaunchKernelGGL((wide_gemm_k<T, BM, BN, TA, TB, PART, STAGES, MAP>), dim3((unsigned)(g.mt * g.nt * g.splits)), dim3(256), lds, s, g);
    return check_launch("wide_gemm");
}

// Tiles of the 16-bit row product.
void rows_tiles(long long N, int K, int NO, int& bm, int& bn) {
    // tiles of 64 rows where 128-row tiles would leave compute units without work
    bm = (long long)cdiv(N, 128) * cdiv(NO, 128) < 256 ? 64 : 128, bn = NO <= 64 ? 64 : 128;
    // 192 columns (a sixth fewer bytes staged per product, longer tiles) where they save a whole round of the 512 tiles
    // that the chip holds; a third longer each ([16384,1152] -> 576, one round instead of two, 35.0 -> 27.4 us; 576 ->
    // 1152, two instead of three, 32.7 -> 29.8; [100000,192] -> 384, four instead of five, would be 31.1 -> 35.7)
    auto rounds = [&](int n) { return cdiv((long long)cdiv(N, 128) * cdiv(NO, n), 512); };
    if (bm == 128 && bn == 128 && K >= 256 && rounds(192) * 4 < rounds(128) * 3) bn = 192;
}

// Tiles and row ranges of the weight gradient: tiles of 64 where a width is no more than that, and the number of ranges whose product by
// itself and with the input gradient, in the launch that they share (both make the same ranges, so that their results are the same), are
// estimated to end first, the latter counting twice.  By itself a compute unit's stages, less each where workgroups take turns.  The shared launch,
// where it is all on the chip at once: the most that a unit is dealt, in order and the ranges first; else all work evenly and part of a
// range's and of a row tile's, which are the last ones.  In both the partials, written and read once more in fp32, and the start of a further round.
// Prices fitted to 1320 random layers of 136 to 1152 channels with every number of ranges (us, MI355X): the ranges chosen take 2.1 % longer than the best
// by themselves and 1.9 % in the shared launch, in fp32 3.1 and 1.9 % (there both cannot be had: [1038,704]^T [1038,352] 17.1 and 20.4 us with two
// ranges, 14.3 and 26.4 with three, since a compute unit's matrix pipe serves one workgroup at a time and 256 are a round).
// us by itself and shared, against 512 workgroups with no more partials than are the operands' traffic, and two stages in LDS: bf16
// [2128,920]^T [2128,464] 29.8 -> 15.1, 34.0 -> 16.0, [1568,1024]^T [1568,512] 22.7 -> 14.3, 24.3 -> 15.6, [16384,1152]^T [16384,576] 36.7 -> 38.9, 59.0 -> 60.2;
// fp32 [2002,1032]^T [2002,516] 40.3 -> 31.0, 58.5 -> 53.7, [1000,512]^T [1000,256] 15.4 -> 11.2, 15.7 -> 16.6.  1370 other random layers 1.14 and 1.13
// times as fast in bf16, 1.09 and 1.04 in fp32 (of the shared launches one in 40 is more than 5 % slower in bf16, one in 23 in fp32).
struct WgradPlan {
    int bm, bn, mt, nt, splits;
    long long kper;
};
WgradPlan wgrad_make_plan(long long N, int M, int NO, int es) {
    const bool f32 = es == 4;
    const int bk = kRowBytes / es;
    // us: a result's stage of a compute unit's only workgroup, of one of several, and of the input gradient; a range's partials
    const double area = f32 ? 64 * 64 : 128 * 128, only = (f32 ? 0.6 : 0.52) / area, several = (f32 ? 0.55 : 0.355) / area,
                 row = (f32 ? 0.55 : 0.44) / area, partial = (f32 ? 2.0e-6 : 1.8e-6) * M * NO + (f32 ? 0.03 : 0.005);
    const double uneven = f32 ? 1.0 : 1.3, end = f32 ? 0.25 : 0.4, last = 0.5;   // shares of a unit's most work, a range's, and a row tile's
    const double again = f32 ? 0.6 : 1.0;   // us: the start of another round of workgroups
    const long long resident = f32 ? 1024 : 512;
    // no range longer than its 32-bit offsets reach (operands of more than 2 GiB, widths that alone fill the chip)
    const long long reach = 0x7fffffffLL / ((long long)(M > NO ? M : NO) * es) / 64 * 64, fewest = reach > 0 ? (N + reach - 1) / reach : 1;
    int rm = 64, rn = 64;
    if (!f32) rows_tiles(N, M, NO, rm, rn);
    const long long rows = (long long)cdiv(N, rm) * cdiv(NO, rn);
    const double row_work = (double)cdiv(M, bk) * rm * rn * row;
    auto shared = [&](long long blocks, double work) {   // (without the partials)
        const long long all = blocks + rows;
        const double even = (blocks * work * several + rows * row_work) / 256;
        if (all > resident) return even + end * work * several + last * row_work + again * (cdiv(all, resident) - 1);
        double most = 0;
        for (const long long unit : {0LL, blocks % 256, all % 256}) {   // (units alike up to the next of these)
            const long long ranges = (blocks + 255 - unit) / 256, n = (all + 255 - unit) / 256;
            most = std::max(most, (ranges * work * several + (n - ranges) * row_work) * (n == 1 ? only / several : 1.0));
        }
        return std::max(even, most * uneven);
    };
    struct Choice {
        WgradPlan p;
        double alone;
    };
    auto best_of = [&](int bm, int bn) {
        Choice best{};
        double least = 0;
        const long long mt = cdiv(M, bm), nt = cdiv(NO, bn), tiles = mt * nt, most = std::max(fewest, std::min(N / 64, 1024 / tiles));
        const bool paired = f32 ? bm == 64 && bn == 64 : bm == 128 && bn == 128;
        for (long long s = fewest; s <= most || s == fewest; s += s < 16 ? 1 : s / 8) {
            const long long kper = ((N + s - 1) / s + 63) / 64 * 64, n = (N + kper - 1) / kper, blocks = tiles * n;
            const double work = (double)(kper / bk) * bm * bn;
            const double alone = work * (blocks <= 256 ? only : cdiv(blocks, 256) * several) + again * (cdiv(blocks, resident) - 1) + partial * n;
            const double cost = paired ? 0.5 * alone + shared(blocks, work) + partial * n : alone;
            if (best.p.splits != 0 && cost >= least) continue;
            least = cost;
            best = {{bm, bn, (int)mt, (int)nt, (int)n, kper}, alone};
        }
        return best;
    };
    const Choice large = best_of(M <= 64 ? 64 : 128, NO <= 64 ? 64 : 128);
    if (!f32) return large.p;
    // fp32, bound by the matrix pipe and not by what the tiles read: tiles of 64 (which the shared launch takes) unless larger ones
    // are clearly faster by themselves, which is one layer in 150 (us, 64 x 64 and larger: [848,780]^T [848,448] 23.8 and 21.0, [939,948]^T
    // [939,348] 25.3 and 20.9, [1496,1088]^T [1496,1136] 57.4 and 48.0, [5951,968]^T [5951,4] 18.0 and 13.8)
    const Choice small = best_of(64, 64);
    return small.alone > 1.15 * large.alone ? large.p : small.p;
}

// (asked for five times a call, the workspace's size among them, and microseconds to make)
WgradPlan wgrad_plan(long long N, int M, int NO, int es) {
    static PlanCache<std::array<long long, 4>, WgradPlan> plans;
    return plans.get({N, M, NO, es}, [=] { return wgrad_make_plan(N, M, NO, es); });
}

// Column sums that ride behind `blocks` workgroups of products: as many workgroups as by themselves, which read while the products multiply.  (192 of them
// are one or two more to a compute unit, but their longer chains outlast the products: us of both launches with the gates', by themselves, 192 and
// all, 418 random 16-bit layers of 8 MB and more 21.2, 20.7 and 20.2 ms, 152 fp32 ones 10.2, 9.7 and 9.5; [65,33,44,280] fp16 84, 94 and 82.)  In 16 bits, where
// a launch of one workgroup a compute unit (kDeep) leaves 64 units or more, no more than those, so that its products keep their four stages: us of the first
// layer, nine of 144 to 180 tiles, by themselves 126, with all 98, with these 87.  (Weights packed beside them make it two stages all the same: [3,14,14,920]
// bf16 15.6 -> 15.4, [12,14,14,920] 15.6 -> 14.7.)
ColsumJob riding_sums(const ColsumJob& j, long long blocks, int es) {
    const long long spare = 256 - blocks;
    if (es == 4 || spare < 64 || colsum_workgroups(j) <= spare) return j;
    const int n = (int)spare, each = j.B * j.slices;
    ColsumJob r = colsum_plan(j.x, j.part, j.B, j.P, j.C, es, n > each ? n - each + 1 : 1);
    r.pairs = r.len > j.len;
    return r;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace

bool dense_wide_ok(int K, int NO, int dtype) {
    const int v = dtype == kF32 ? 4 : 8;   // values of 16 bytes
    return K >= v && NO >= v && K % v == 0 && NO % v == 0;
}

// Arguments and tiles of the row product; false: not covered (widths, alignment, offsets of 2^31 bytes within a tile or a weight).
static bool wide_rows_plan(WideArgs& g, int& bm, int& bn, const void* x, const void* w, int w_kmajor, const void* bias, const float* rowbias,
                           void* y, long long N, int K, int NO, int P, int dtype) {
    const int es = dtype == kF32 ? 4 : 2;
    if (!dense_wide_ok(K, NO, dtype) || N > 0x7fffffffLL || (long long)K * NO * es > 0x7fffffffLL || K > (1 << 21) || NO > (1 << 21))
        return false;
    if (!aligned16(x) || !aligned16(w) || !aligned16(y) || !aligned16(rowbias) || (reinterpret_cast<uintptr_t>(bias) & (es == 4 ? 15 : 7)))
        return false;
    g = WideArgs{x, w, bias, rowbias, y, N, K, NO, K, w_kmajor ? NO : K, P > 0 ? P : 1, 0, 0, 1, (long long)cdiv(K, 64) * 64};
    if (es == 4) {
        // small tiles, four to a compute unit ([100352,128] -> 64: 22.8 us, 128 x 64 26.9, 128 x 128 41.7; never slower where
        // it matters), but not for many rows of a short sum, which is a stream ([50000,16] -> 32: 6.4 here, 5.6 in dense_any.hip)
        if (K < 32 && N >= 16384 && NO <= 256) return false;
        bm = bn = 64;
    } else {
        rows_tiles(N, K, NO, bm, bn);
    }
    g.mt = cdiv(N, bm), g.nt = cdiv(NO, bn);
    return (long long)g.mt * g.nt <= 0x7fffffffLL;
}

// -1: not covered.
int dense_wide_rows_launch(const void* x, const void* w, int w_kmajor, const void* bias, const float* rowbias, void* y,
                           long long N, int K, int NO, int P, int dtype, hipStream_t s, const RowMap* map) {
    WideArgs g;
    int bm, bn;
    if (map && (w_kmajor || dtype == kF32)) return -1;
    if (!wide_rows_plan(g, bm, bn, x, w, w_kmajor, bias, rowbias, y, N, K, NO, P, dtype)) return -1;
    if (N == 0) return 0;
    if (map) g.map = *map;
#define PDW_WIDE_S(T, BM, BN, STAGES)                              \
    (w_kmajor ? wide_go<T, BM, BN, false, true, false, STAGES>(g, s) \
     : map    ? wide_go<T, BM, BN, false, false, false, STAGES, true>(g, s) : wide_go<T, BM, BN, false, false, false, STAGES>(g, s))
#define PDW_WIDE_T(T, BM, BN) PDW_WIDE_S(T, BM, BN, kDeep)
#define PDW_WIDE(BM, BN) (dtype == kF16 ? PDW_WIDE_T(f16_t, BM, BN) : PDW_WIDE_T(bf16_t, BM, BN))
#define PDW_WIDE2(BM, BN) (dtype == kF16 ? PDW_WIDE2_T(f16_t, BM, BN) : PDW_WIDE2_T(bf16_t, BM, BN))   /* (tiles of launches that fill the chip) */
#define PDW_WIDE2_T(T, BM, BN) PDW_WIDE_S(T, BM, BN, 2)
    if (dtype == kF32) return w_kmajor ? wide_go<float, 64, 64, false, true, false, 2>(g, s) : wide_go<float, 64, 64, false, false, false, 2>(g, s);
    if (bn == 192) return PDW_WIDE2(128, 192);
    if (bm == 64) return bn == 64 ? PDW_WIDE(64, 64) : PDW_WIDE(64, 128);
    return bn == 64 ? PDW_WIDE2(128, 64) : PDW_WIDE2(128, 128);
#undef PDW_WIDE
#undef PDW_WIDE2
#undef PDW_WIDE_T
#undef PDW_WIDE2_T
#undef PDW_WIDE_S
}

namespace {

template <typename T, int BM, int BN, int STAGES>
int first_go(const WideArgs& g, const QuadArgs& qa, const ColsumJob& sums, const PackArgs* pack, hipStream_t s) {
    constexpr size_t stages = wide_lds<T, BM, BN, false, STAGES>(), red = 256 * 16 / sizeof(T) * sizeof(float), lds = stages > red ? stages : red;
    const long long nrows = (long long)g.mt * g.nt, nsums = colsum_workgroups(sums), all = nrows + nsums + (pack ? pack_workgroups(*pack) : 0);
    if (all > 0x7fffffffLL) return -1;
    if constexpr (STAGES == kDeep) {
        if (!goes_deep<T>(all, lds, g.Kd, 6)) return first_go<T, BM, BN, 2>(g, qa, sums, pack, s);
    }
    if constexpr (lds > 64 * 1024) {
        static std::once_flag once;
        std::call_once(once, [] {
            (void)hipFuncSetAttribute((const void*)wide_first_k<T, BM, BN, STAGES>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
            if constexpr (sizeof(T) == 2) (void)hipFuncSetAttribute((const void*)wide_first_pack_k<T, BM, BN, STAGES>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        });
    }
    if constexpr (sizeof(T) == 2) {
        if (pack) {
            hipLaunchKernelGGL((wide_first_pack_k<T, BM, BN, STAGES>), dim3((unsigned)all), dim3(256), lds, s, g, qa, sums, (int)nrows, (int)nsums, *pack);
            return check_launch("wide_first_pack");
        }
    }
    hipLaunchKernelGGL((wide_first_k<T, BM, BN, STAGES>), dim3((unsigned)all), dim3(256), lds, s, g, qa, sums, (int)nrows);
    return check_launch("wide_first");
}

}  // namespace

// Whether dense_wide_first_launch takes the layer (its plan for the sums in *sums, without pointers).
bool dense_wide_first_plan(ColsumJob* sums, long long N, int K, int NO, int B, int P, int dtype) {
    const int es = dtype == kF32 ? 4 : 2;
    WideArgs g;
    int bm, bn;
    alignas(16) static char any[16];
    if (N < 1 || !wide_rows_plan(g, bm, bn, any, any, 0, nullptr, nullptr, any, N, K, NO, P, dtype)) return false;
    *sums = riding_sums(colsum_plan(nullptr, nullptr, B, P, K, es), (long long)g.mt * g.nt, es);
    return true;
}

// y[N][NO] = x W^T, W stored [NO][K] or, with pack, as given there (zero rows where the layout has padding), the column sums of x as
// planned, and in pool the means of the 2 x 2 pixels of y, images of 2 w_half columns; -1: not covered.
int dense_wide_first_launch(const void* x, const void* w, void* y, void* pool, int w_half, long long N, int K, int NO, const ColsumJob& sums,
                            const PackArgs* pack, int dtype, hipStream_t s) {
    WideArgs g;
    int bm, bn;
    const int es = dtype == kF32 ? 4 : 2;
    if (N < 1 || (pack && dtype == kF32) || !wide_rows_plan(g, bm, bn, x, w, 0, nullptr, nullptr, y, N, K, NO, 1, dtype)) return -1;
    // a tile of rows by quads reaches 32 quads and two pairs of image rows far: 32-bit offsets
    if (!aligned16(pool) || (N & 3) || w_half < 1 || w_half > 32768 || (128LL + 8 * w_half) * K * es > 0x7fffffffLL) return -1;
    if (pack) g.map = RowMap{pack->Gp, pack->G};
    const QuadArgs qa{pool, w_half, w_half > 1 ? (uint32_t)((0x100000000ULL + w_half - 1) / w_half) : 0u};
    auto go = [&](auto t) {
        using T = decltype(t);
        if (bn == 192) return first_go<T, 128, 192, 2>(g, qa, sums, pack, s);
        if (bm == 64) return bn == 64 ? first_go<T, 64, 64, kDeep>(g, qa, sums, pack, s) : first_go<T, 64, 128, kDeep>(g, qa, sums, pack, s);
        return bn == 64 ? first_go<T, 128, 64, 2>(g, qa, sums, pack, s) : first_go<T, 128, 128, 2>(g, qa, sums, pack, s);
    };
    if (dtype == kF32) return first_go<float, 64, 64, 2>(g, qa, sums, nullptr, s);
    return dtype == kF16 ? go(f16_t{}) : go(bf16_t{});
}

// (of either type)
size_t dense_wide_wgrad_workspace(long long N, int M, int NO) {
    if (N < 1 || M < 1 || NO < 1) return 0;
    const int a = wgrad_plan(N, M, NO, 2).splits, b = wgrad_plan(N, M, NO, 4).splits;
    return (size_t)(a > b ? a : b) * M * NO * sizeof(float);
}

int dense_wide_wgrad_launch(const void* a, const void* b, void* dw, void* ws, long long N, int M, int NO, int dtype, hipStream_t s) {
    if (!dense_wide_ok(M, NO, dtype) || N < 1 || !aligned16(a) || !aligned16(b) || !aligned16(ws)) return -1;
    const int es = dtype == kF32 ? 4 : 2;
    // (fp32 widths up to 256: one 32 x 32 tile a wavefront, dense_any.hip, needs no LDS and is as fast or faster, [100352] rows of
    // 128 x 64 24.3 us with its summation against 27.9, [784] of 248 x 124 7.1 against 9.6)
    if (es == 4 && M <= 256 && NO <= 256) return -1;
    const WgradPlan p = wgrad_plan(N, M, NO, es);
    if (p.kper * (M > NO ? M : NO) * es > 0x7fffffffLL) return -1;
    WideArgs g{a, b, nullptr, nullptr, ws, M, N, NO, M, NO, 1, p.mt, p.nt, p.splits, p.kper};
#define PDW_WIDE_W(BM, BN)                                                 \
    (dtype == kF32   ? wide_go<float, BM, BN, true, true, true, 2>(g, s)   \
     : dtype == kF16 ? wide_go<f16_t, BM, BN, true, true, true>(g, s)      \
                     : wide_go<bf16_t, BM, BN, true, true, true>(g, s))
    const int e = p.bm == 64 ? (p.bn == 64 ? PDW_WIDE_W(64, 64) : PDW_WIDE_W(64, 128))
                             : (p.bn == 64 ? PDW_WIDE_W(128, 64) : PDW_WIDE_W(128, 128));
#undef PDW_WIDE_W
    if (e) return e;
    if (dtype == kF32) return wgrad_reduce_launch<float>((const float*)ws, dw, p.splits, M * NO, s);
    if (dtype == kF16) return wgrad_reduce_launch<f16_t>((const float*)ws, dw, p.splits, M * NO, s);
    return wgrad_reduce_launch<bf16_t>((const float*)ws, dw, p.splits, M * NO, s);
}

// Whether the column sums j of the gradient of a layer with NO inputs are best made by workgroups of their own in the launch of both its gradients, which is bound
// by its matrix products more than by memory, instead of that of the gates, which has other bytes to move: where it is large, and twice that where 16-bit
// products fill no more than one round of 512 workgroups, whose tiles were cut to end together and which the sums then outlast.  us of the two launches: [32,56,56,128]
// fp32 (51 MB) 65.9 -> 61.5, [4,64,64,1152] fp16 (38 MB) 81.7 -> 79.5, [8,112,112,256] bf16 (51 MB) 58.4 -> 55.9, [104,27,28,280] 68.6 -> 66.9, [8,48,48,256] fp32
// (19 MB) 40.3 -> 37.8; [2,40,40,640] bf16 (4.1 MB) 17.6 and 17.9, [3,25,20,920] (2.8 MB) 20.3 and 20.5.  Sums over random 16-bit layers, ms: 8 to 17 MB, one round 116 of
// them 3.07 and 3.06 (15 of them slower by 1 to 2.5 % of their step), more 116 of them 3.66 -> 3.51; 17 to 33 MB, one round 47 of them 1.63 -> 1.58, more 140 of them 6.13 -> 5.87; more
// than 33 MB 163 of them 13.5 -> 12.8.
bool dense_wide_sums_ride(const ColsumJob& j, int NO, int dtype) {
    const int es = dtype == kF32 ? 4 : 2;
    const long long N = (long long)j.B * j.P, bytes = N * j.C * es, large = 8 << 20;
    if (bytes < large || bytes >= 2 * large || es == 4) return bytes >= large;
    const WgradPlan p = wgrad_plan(N, j.C, NO, es);
    int bm, bn;
    rows_tiles(N, j.C, NO, bm, bn);
    return (long long)p.mt * p.nt * p.splits + (long long)cdiv(N, bm) * cdiv(NO, bn) > 512;
}

// dx[N,NO] = gy[N,M] W (+ rowbias), W stored [M][NO], and dW[M][NO] = gy^T b, in one launch; -1: not covered, or products that
// other kernels make (the caller makes them one by one).  max_chunks: partials the workspace holds.
// sums (optional): of gy, planned here within what it was given as.
int dense_wide_bwd_pair_launch(const void* gy, const void* w, const void* b, void* dx, void* dw, void* ws, const float* rowbias, int P,
                               long long N, int M, int NO, int dtype, int max_chunks, hipStream_t s, ColsumJob* sums) {
    WideArgs rows, wg{};
    AnyWgradArgs any{};
    int bm, bn, nw, nparts;
    if (N < 1 || !aligned16(b) || !aligned16(ws) || !dense_wide_ok(M, NO, dtype)) return -1;
    if (!wide_rows_plan(rows, bm, bn, gy, w, 1, nullptr, rowbias, dx, N, M, NO, P, dtype)) return -1;
    const int es = dtype == kF32 ? 4 : 2;
    WgradPlan p{};
    const bool small = es == 4 && M <= 256 && NO <= 256;   // (as dense_wide_wgrad_launch chooses)
    if (small) {
        if (!any_wgrad_args(any, gy, b, ws, N, M, NO, dtype, max_chunks)) return -1;
        nw = any.chunks * any_wgrad_groups(any), nparts = any.chunks;
    } else {
        p = wgrad_plan(N, M, NO, es);
        if (p.kper * (M > NO ? M : NO) * es > 0x7fffffffLL) return -1;
        wg = WideArgs{gy, b, nullptr, nullptr, ws, M, N, NO, M, NO, 1, p.mt, p.nt, p.splits, p.kper};
        nw = p.mt * p.nt * p.splits, nparts = p.splits;
    }
    ColsumJob riding{};
    if (sums) riding = riding_sums(*sums, nw + (long long)rows.mt * rows.nt, es);
    const ColsumJob* const ride = sums ? &riding : nullptr;
    int e = -1;
    if (es == 4) {
        if (small) e = pair_go<float, 64, 64, 0, 0, 2>(rows, wg, any, nw, ride, s);
        else if (p.bm == 64 && p.bn == 64) e = pair_go<float, 64, 64, 64, 64, 2>(rows, wg, any, nw, ride, s);
    } else if (p.bm == 128 && p.bn == 128) {
        auto go = [&](auto t) {
            using T = decltype(t);
            if (bn == 192) return pair_go<T, 128, 192, 128, 128, 2>(rows, wg, any, nw, ride, s);
            if (bm == 64 && bn == 128) return pair_go<T, 64, 128, 128, 128, kDeep>(rows, wg, any, nw, ride, s);
            if (bm == 128 && bn == 128) return pair_go<T, 128, 128, 128, 128, 2>(rows, wg, any, nw, ride, s);
            return -1;
        };
        e = dtype == kF16 ? go(f16_t{}) : go(bf16_t{});
    }
    if (e) return e;
    if (sums) *sums = riding;   // (where no kernel takes the layer the caller's plan stands)
    if (dtype == kF32) return wgrad_reduce_launch<float>((const float*)ws, dw, nparts, M * NO, s);
    if (dtype == kF16) return wgrad_reduce_launch<f16_t>((const float*)ws, dw, nparts, M * NO, s);
    return wgrad_reduce_launch<bf16_t>((const float*)ws, dw, nparts, M * NO, s);
}

}  // namespace pdw
