// Depthwise convolution as a block-Toeplitz product on the dense matrix cores: forward and input gradient for
// 16-bit types, stride 1, dilation 1, odd square filters up to 17 (the input gradient is the same kernel run on gy
// with the 180-degree rotated filter and padding k-1-p).
//
// For one channel, a patch of 4 x 4 outputs is a product of the filter, spread out as a 16 x (K+3)(K+3) matrix
//     A[(di,dj)][(r,s)] = w[r - di][s - dj]          (zero where the tap falls outside the filter)
// with the patch's (K+3) x (K+3) input window as a vector.  v_mfma_f32_16x16x32_{bf16,f16} computes
// D[m][n] += sum_k A[m][k] B[k][n] with m = one of the patch's 16 outputs, n = one of 16 patches and k running over
// 32 window positions per instruction: 4 "k groups" of 8 consecutive columns of one window row, which is what one
// lane holds (lane = n + 16 * group for B, m + 16 * group for A).  A window row is ICB = ceil((K+3)/8) groups wide,
// so a patch takes NM = ceil((K+3) * ICB / 4) instructions (8 at K = 13: 169 of every 256 multiply-adds fall on a
// real tap, on the pipe that runs at four times the rate of the 4x4x4 block form).  A depends on the channel only:
// each wavefront owns CPW channels and keeps their A operands in registers for the whole kernel.
//
// The 16 patches of an instruction lie side by side (4 columns apart) in NI = 16 / NPC images, and a wavefront
// walks down the rows four at a time.  Moving down by 4 rows shifts every B operand by ICB instructions, so the
// operands live in a register ring: a step reads only the 4 new window rows from LDS (ICB operands of 16 bytes per
// lane) for NM instructions.  That is what makes the kernel a stream: per step and channel 2 LDS reads, 8 MFMAs.
//
// A workgroup (8 wavefronts, CS = 8 CPW channels) owns 4 NPC columns of NI images side by side and a run of output rows.  The
// images of a batch are stacked into one column of rows, `per` rows apart with zeros between them, and a run starts and ends
// anywhere (at multiples of 8 rows): as many workgroups as the chip holds at once, whatever the extents, each with one
// start-up.  There are at least PH rows of zeros, and more where the last patch of an image needs them: its operands cover
// OPR >= K + 3 window rows, of which those beyond the K + 3 (and those below an image's last output) meet zeros of A, and zero
// times an infinity of the next image would be NaN.  Runs that are parts of one image read nothing of another.  The input window is streamed through LDS, channel-major: xl[image][channel][row][column] as 16-bit
// values, so that 8 consecutive columns of a channel are 16 contiguous bytes.  Threads load 4 pixels of a row x 8 channels (four
// 16-byte loads), interleave columns with byte permutes and write 8 bytes per channel; the passes of this copy are requested two
// ahead and committed only as far as the next step needs.  Results are rounded once, transposed through a small
// double-buffered LDS tile (pixel-major, one dword of padding per 4 pixels keeps the 4-byte scatter free of bank conflicts) and
// leave as 16-byte stores, one step behind the MFMAs.
//
// What bounds it: the instructions that move data, and waiting.  By the counters ([128,56,56,64] filter 13, 47 k cycles) the LDS is
// busy 41 % of the cycles, the matrix pipe 33 and the vector ALU 31, and a wavefront, two to a SIMD, waits for data or a barrier a
// third of its time and for its turn to issue another third.  Hence rows are counted with scalars (images a multiple of 8 rows
// apart, so that a step or pass meets a boundary as a whole), LDS writes are 8 bytes with constant offsets, and the pieces that
// move data are written between the products.  115 vector instructions a step became 64 and [8,56,56,64], filter 13, in 8 long
// runs 1.15 us a step 0.97; what does not overlap yet is the LDS round trips either side of the barrier.
//
// MODE is a set of bits.
// 1 (input gradient of a tensor that was also average-pooled 2x2): y += add[i/2, j/2] / 4 in the store; 16: that of a pool
// of any ratio down to AH x AW, from the at most 2 x 2 bins that a pixel lies in.
// 2 (forward): the 2x2 average pool of x is written to `pool` by the staging threads, which hold exactly the
// four pixels of a pool window in registers (needs even padding, so that windows do not straddle threads).
// 4 (forward, inference): the gate of conv_block.py:18-19 in the store.  A workgroup's 16 channels are 8 of the first
// half and the matching 8 of the second half of C, and the two store threads of a pixel multiply four channel pairs
// each (the rounded convolution outputs, as the stand-alone gate kernel does): y[..., c] = conv[c] * conv[C/2 + c] * gs,
// C/2 channels wide, written with a pixel stride of YC channels from channel `ych` on (into the concatenation).
// With 8 channels per workgroup (filters from 15 on) the slice is 4 channels of each half: every 16-byte load of the
// staging and of the filter becomes two 8-byte loads C bytes apart, and a pixel's one store thread gates the two
// halves of its piece.
// 8: with any of these but the pool, runs of no more than tz_short(K) steps.
//
// Zero entries of A multiply real pixels of the window (and the window is wider than K+3 where (K+3) % 8 != 0), so a
// non-finite input value reaches outputs of its own image up to 3 + 8 ICB - (K+3) pixels beyond its K x K footprint as NaN.
#pragma once
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "tile_common.h"

namespace pdw {

typedef float tz_f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ tz_f32x4 mfma16(uint4 a, uint4 b, tz_f32x4 c, bf16_t) {
    typedef __bf16 v8 __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
}
__device__ __forceinline__ tz_f32x4 mfma16(uint4 a, uint4 b, tz_f32x4 c, f16_t) {
    typedef _Float16 v8 __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
}

template <int K, int NPC, int CS>
struct TzShape {
    static constexpr int NT = 512, NWV = 8;
    static constexpr int IC = K + 3;                  // window columns (and rows) of a 4 x 4 patch
    static constexpr int ICB = (IC + 7) / 8;          // k groups per window row
    static constexpr int NKG = IC * ICB;              // k groups of a patch
    static constexpr int NM = (NKG + 3) / 4;          // MFMAs per patch (group of 16) and channel
    static constexpr int PER = (NM + ICB - 1) / ICB;  // row groups (of 4 rows) an operand ring spans
    static constexpr int OPR = (4 * NM + ICB - 1) / ICB;  // window rows that a patch's operands cover (those from IC on meet zeros of A)
    static constexpr int RING = PER * ICB;            // operands in the ring
    static constexpr int NI = 16 / NPC;               // images side by side in one instruction
    static constexpr int TW = 4 * NPC;                // output columns of a workgroup
    static constexpr int NH = CS / 8;                 // 8-channel pieces per pixel
    static constexpr int CPW = CS / NWV;              // channels per wavefront
    static constexpr int PIECES = TW * 4 * NI * NH;   // 16-byte pieces of a result tile
    static constexpr int TPT = NT / PIECES < 2 ? 1 : 2, NG = 2 / TPT;   // tiles stored side by side, and one after the other
    static constexpr int WCOLS = 4 * (NPC - 1) + 8 * ICB;  // window columns the operands touch
    static constexpr int RP = (2 * WCOLS + 7) / 8 * 8;     // bytes per window row of a channel
    static constexpr int OPX = 2 * CS;                     // bytes per pixel of the result tile
    static constexpr int OROWP = TW * OPX + NPC * 4;       // bytes per row of the result tile (4 per 4 pixels padding)
    static constexpr int OLB = NI * 4 * OROWP;             // one result tile: 4 rows of every image
    static constexpr int WTH = 4 * PER + 3, WTW = 8 * ICB + 4;  // zero-bordered filter table [channel][WTH][WTW]
    static constexpr int WTB = CS * WTH * WTW * 2;
    static constexpr int R2B = (4 * OLB > 2 * WTB ? 4 * OLB : 2 * WTB + 15) / 16 * 16;  // 4 result tiles / two filter tables (shared)
    static_assert(K % 2 == 1 && K >= 3 && K <= 17, "odd filters up to 17");
    static_assert(NPC == 16 || NPC == 8, "patches per image row");
    static_assert(CS == 8 || CS == 16, "channels per workgroup");
    // The window lives in LDS as a ring of NR row groups (of 4 rows), window row r at ring row r % NRR: a step reads
    // the two row groups it adds to the operand registers while the next step's two are being written, and the
    // first step needs PER + 1 row groups in place before it starts.
    static constexpr int NR = PER + 1 > 4 ? PER + 1 : 4;
    static constexpr int NRR = 4 * NR;
    static constexpr int CHP = NRR * RP % 16 == 8 ? NRR * RP : NRR * RP + 8;  // bytes per channel plane, = 8 mod 16
    static_assert(CHP == NRR * RP + 8, "the spare bytes of a plane");
    // Where staging lanes without an item write, 8 planes apart like an item: the 8 bytes behind a plane's rows, which nobody reads;
    // where the pool is written, whose items are two rows, space of its own behind the result tiles.  (With that everywhere a workgroup
    // of filters 3 and 5, 64 columns wide, had no room for a second one beside it: launches of 257 .. 512 workgroups took 1.13 times as
    // long, of up to 1024 1.2, beyond 1.36.)
    static constexpr int ENDS = NI * CS * CHP + R2B;
    static constexpr int spare(bool pool) { return pool ? ENDS : NRR * RP; }
    static constexpr int bins_at = (ENDS + 15) / 16 * 16;   // (MODE & 16) 8 bytes an output row
    static constexpr size_t lds_bytes = ENDS, lds_bytes_pool = (size_t)ENDS + 7 * CHP + RP + 16;
    static_assert(lds_bytes_pool <= 160 * 1024, "LDS");
    static_assert(K > 5 || lds_bytes <= 80 * 1024, "two workgroups on a compute unit");
};

// 2^32 / d rounded up (0 for 1): n / d = the high half of n times this while n d < 2^32.  (A division costs a wavefront about
// 150 cycles, and a workgroup cannot request its first rows before it has made a handful.)
inline uint32_t tz_inverse(int d) { return d == 1 ? 0u : (uint32_t)(((1ULL << 32) + d - 1) / (uint32_t)d); }
// Rows to the next image for a run that knows its own only: further than it reaches, and the inverse that makes all of its rows
// lie in image 0 (n * 1 / 2^32).
constexpr int kTzAlone = 0x40000000;
constexpr uint32_t kTzAloneInverse = 1;
__device__ __forceinline__ int tz_quotient(int n, uint32_t inverse) { return inverse ? (int)__umulhi((uint32_t)n, inverse) : n; }

// How a problem is cut into workgroups (tz_cut).
struct TzRuns {
    int per;           // rows from one image to the next in the stack of a batch's images (a multiple of 8); kTzAlone if rpi
    int run;           // stacked rows of a workgroup (a multiple of 8)
    int rpi;           // 0: runs follow one another through the stack; else they are parts of an image, rpi of them to one
    int nruns;         // (0: not covered)
    uint32_t per_inv, rpi_inv, ncolt_inv, nslices_inv;   // tz_inverse of these
};

struct TzGeom : TzRuns {
    int B, H, W, C;    // input extents
    int OH, OW;        // output extents
    int PH, PW;        // padding
    int ncolt, nslices;
    int stack;         // (host) rows from one image to the next in the stack (0: no stack)
    int flip;          // 1: 180-degree rotated filter (input gradient)
    int AH, AW;        // extents of the half-resolution addend / pooled output
    int YC, ych;       // output pixel stride in channels, first output channel
    float gs;          // gate factor (MODE & 4)
};

// 8 values of T: a + b / 4, rounded once more (what an accumulating pool gradient does to a stored tensor).
template <typename T>
__device__ __forceinline__ uint4 tz_add_quarter(uint4 a, uint4 b) {
    union U {
        uint4 u;
        T t[8];
    } ua, ub, uo;
    ua.u = a, ub.u = b;
#pragma unroll
    for (int i = 0; i < 8; ++i) uo.t[i] = from_f32<T>(to_f32(ua.t[i]) + 0.25f * to_f32(ub.t[i]));
    return uo.u;
}

// 8 values of T: a + the weighted gradients of up to four bins, rounded once more: avgpool_bwd_k's sum to the bit (bins that are not there are
// zeros).
template <typename T>
__device__ __forceinline__ uint4 tz_add_bins(uint4 a, const uint4 (&b)[4], float w0, float w1, float w2, float w3) {
    union U {
        uint4 u;
        T t[8];
    } ua, ub[4], uo;
    ua.u = a;
#pragma unroll
    for (int k = 0; k < 4; ++k) ub[k].u = b[k];
#pragma unroll
    for (int i = 0; i < 8; ++i)
        uo.t[i] = from_f32<T>(to_f32(ua.t[i]) + fmaf(to_f32(ub[3].t[i]), w3, fmaf(to_f32(ub[2].t[i]), w2, fmaf(to_f32(ub[1].t[i]), w1, fmaf(to_f32(ub[0].t[i]), w0, 0.f)))));
    return uo.u;
}

// 4 values of T: a * b * s, rounded once (the arithmetic of the stand-alone gate kernel).
template <typename T>
__device__ __forceinline__ uint2 tz_gate(uint2 a, uint2 b, float s) {
    union U {
        uint2 u;
        T t[4];
    } ua, ub, uo;
    ua.u = a, ub.u = b;
#pragma unroll
    for (int i = 0; i < 4; ++i) uo.t[i] = from_f32<T>(gate_f32(to_f32(ua.t[i]), to_f32(ub.t[i]), s));
    return uo.u;
}

// Steps of a run up to which MODE 8 is there (0: never).  A run's last steps request passes past its window, which move nothing
// but take their turn at the address unit, in front of the run's result stores; left out as constants, since with a branch the compiler
// no longer knows which requests are the newest, and not beside the general code, which then has 36 registers more (us: [108,10,13,40]
// filter 5, two steps, 5.8 -> 5.3, [2,33,44,440] filter 3 6.0 -> 5.6; [18,7,7,224] filter 15, one step, 6.45 -> 5.95, [4,8,10,176]
// filter 17 6.15 -> 6.05; with bands of one image, which requested nothing past a window, 5.35, 5.65, 6.15 and 6.0).
constexpr int tz_short(int K) { return K <= 5 ? 2 : K >= 15 ? 1 : 0; }

// f(0), f(1), ... f(N - 1) with constants, until one of them answers false.
template <int J, int N, typename F>
__device__ __forceinline__ void tz_in_turn(F& f) {
    if constexpr (J < N) {
        if (f(std::integral_constant<int, J>())) tz_in_turn<J + 1, N>(f);
    }
}

// One workgroup's run: `blk` of the problem's `nblk` workgroups.
template <typename T, int K, int NPC, int CS, int MODE>
__device__ __forceinline__ void dwconv_tz_body(const T* __restrict__ x, const T* __restrict__ w,
                                               const T* __restrict__ add, T* __restrict__ pool, T* __restrict__ y,
                                               const TzGeom& g, int blk, int nblk) {
    using Sh = TzShape<K, NPC, CS>;
    constexpr int NT = Sh::NT, NG = Sh::NG, ICB = Sh::ICB, NKG = Sh::NKG, NM = Sh::NM, PER = Sh::PER, RING = Sh::RING;
    constexpr int NI = Sh::NI, TW = Sh::TW, NH = Sh::NH, CPW = Sh::CPW, RP = Sh::RP, OPX = Sh::OPX, OROWP = Sh::OROWP;
    constexpr int OLB = Sh::OLB, WTH = Sh::WTH, WTW = Sh::WTW, NR = Sh::NR, NRR = Sh::NRR, CHP = Sh::CHP;
    constexpr bool ANY = (MODE & 16) != 0, ADD = (MODE & 1) != 0 || ANY, POOL = (MODE & 2) != 0, GATE = (MODE & 4) != 0;
    constexpr int SHORT = (MODE & 8) != 0 ? tz_short(K) : 0, PASSES = SHORT ? SHORT + 1 : 4;   // steps of a run at most; passes before them
    static_assert(!GATE || !ADD, "the gate is a forward mode");
    static_assert(!(SHORT && POOL), "short runs do not write the pool");
    // the gate pairs channel c with channel C/2 + c: a 16-channel slice is 8 channels of each half of C (its two
    // 8-channel pieces), an 8-channel slice 4 of each (the halves of its one piece, moved as two 8-byte accesses)
    constexpr bool G8 = GATE && CS == 8;
    static_assert(!(G8 && POOL), "the pool's stores assume 8 contiguous channels");
    extern __shared__ uint32_t smem[];
    char* const xl = reinterpret_cast<char*>(smem);        // [NI][CS] planes of CHP bytes: [ring row][column] of T
    char* const r2 = xl + NI * CS * CHP;                 // filter table, then the two result tiles

    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    int bid = xcd_remap(blk, nblk);
    int rest = tz_quotient(bid, g.nslices_inv);
    const int sl = bid - rest * g.nslices;
    bid = tz_quotient(rest, g.ncolt_inv);
    const int ct = rest - bid * g.ncolt;
    const int c0 = sl * CS, ocol0 = ct * TW;
    auto images_in = [&](int v) { return tz_quotient(v, g.per_inv); };   // (v >= 0)
    // the run's output rows: a part of an image, or g.run of the stack without the rows between images at its ends
    int b0, orow0, rows_valid;
    if (g.rpi) {
        const int image = tz_quotient(bid, g.rpi_inv);
        orow0 = (bid - image * g.rpi) * g.run, rows_valid = min(g.run, g.OH - orow0), b0 = image * NI;
    } else {
        const int first = bid * g.run;
        b0 = images_in(first), orow0 = first - b0 * g.per;
        int end = orow0 + min(g.run, ((g.B + NI - 1) / NI - 1) * g.per + g.OH - first);   // (from image b0's first row on)
        if (orow0 >= g.OH) ++b0, orow0 = 0, end -= g.per;
        if (end <= 0) return;     // (uniform) all of them between two images
        const int over = images_in(end - 1) * g.per;
        rows_valid = min(end, over + g.OH) - orow0;
        b0 *= NI;
    }
    const int cols_valid = min(TW, g.OW - ocol0);
    const int nsteps = (rows_valid + 3) >> 2;
    const int NROWS = 4 * (nsteps + PER - 1);              // window rows the steps read
    const long long img_in = (long long)g.H * g.W * g.C, img_out = (long long)g.OH * g.OW * g.YC;
    // first channel of the slice's 8-channel piece h
    auto chof = [&](int h) { return G8 ? 4 * sl : GATE ? 8 * sl + h * (g.C >> 1) : c0 + 8 * h; };

    // ---- filter slice, 8 channels of a tap per load: requested before the window, so that waiting for it leaves
    // the window's loads in flight
    constexpr int NWL = (K * K * NH + NT - 1) / NT;
    uint4 wval[NWL];
#pragma unroll
    for (int i = 0; i < NWL; ++i) {
        const int idx = min(tid + i * NT, K * K * NH - 1);
        if constexpr (G8) {
            const T* wp = w + idx * g.C + 4 * sl;
            const uint2 lo = *reinterpret_cast<const uint2*>(wp), hi = *reinterpret_cast<const uint2*>(wp + (g.C >> 1));
            wval[i] = make_uint4(lo.x, lo.y, hi.x, hi.y);
        } else {
            wval[i] = *reinterpret_cast<const uint4*>(w + (idx / NH) * g.C + min(chof(idx % NH), g.C - 8));
        }
    }

    // ---- staging.  The window arrives in passes, requested two ahead into two register buffers.  Passes 0 and 1
    // are halves of the PER + 1 row groups (of 4 rows) the first step reads, every later pass the two row groups the
    // next step adds, so step f is preceded by the commit of pass f + 1.  A thread's item is (IR rows of the pass,
    // image, IC columns cq, 8-channel piece h), h fastest, the same in every pass.
    constexpr int IR = POOL ? 2 : 1, IC = POOL ? 2 : 4;          // (the pool's windows are 2 x 2)
    constexpr int RW01 = 2 * PER + 2;                            // rows of pass 0 and of pass 1
    constexpr int RWMAX = RW01 > 8 ? RW01 : 8;
    constexpr int WCQ = Sh::WCOLS / IC;
    constexpr int NLD = (RWMAX / IR * NI * (Sh::WCOLS / IC) * NH + NT - 1) / NT;  // items per thread and pass
    // A step has too few products to put the staging between them: the previous step's tiles leave before them instead (us:
    // [32,56,56,128] filter 3 14.4 -> 13.4, [64,28,28,256] 15.5 -> 14.8; the tiles behind the staging: 14.6 and 16.4).
    constexpr bool FEW = NM <= 2;
    constexpr int UNRF = PER % 4 == 0 ? PER / 2 : (PER % 2 == 0 ? PER : 2 * PER);  // steps per trip: even, PER | 2 UNRF
    auto first_row = [&](int pass) { return pass < 2 ? pass * RW01 : 2 * RW01 + 8 * (pass - 2); };
    // Loads go through a buffer descriptor over the workgroup's images: an offset past its end (an image beyond the
    // batch, or one of the markers for a row / column / channel outside the tensor) reads as zero and moves no
    // data, which is the zero padding.  The images of a run hold less than 2^29 elements (guarded on the host), so valid
    // byte offsets stay below 2^30 and any sum with a marker stays past the end.
    constexpr uint32_t kNoCol = 0x40000000u, kNoRow = 0x80000000u;
    // images the run reaches (all of its offsets are from b0 on)
    const int images = min((images_in(orow0 + rows_valid + K + 24) + 1) * NI, g.B - b0);
    const __amdgpu_buffer_rsrc_t xrsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<T*>(x + (long long)b0 * img_in), (short)0, (int)(images * img_in * 2), 0x00020000);
    auto xload_from = [&](const __amdgpu_buffer_rsrc_t& r, uint32_t off, uint32_t soff = 0) {
        typedef unsigned v4u __attribute__((ext_vector_type(4)));
        const v4u v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, (int)soff, 0);
        return make_uint4(v.x, v.y, v.z, v.w);
    };
    auto xload = [&](uint32_t off) {
        if constexpr (G8) {   // 4 channels of each half of C (C bytes apart); a marker offset stays past the end
            typedef unsigned v2u __attribute__((ext_vector_type(2)));
            const v2u lo = __builtin_amdgcn_raw_buffer_load_b64(xrsrc, (int)off, 0, 0);
            const v2u hi = __builtin_amdgcn_raw_buffer_load_b64(xrsrc, (int)(off + (uint32_t)g.C), 0, 0);
            return make_uint4(lo.x, lo.y, hi.x, hi.y);
        } else {
            return xload_from(xrsrc, off);
        }
    };
    uint32_t icol[NLD][IC];  // byte offsets of the item's columns (image and channel piece included), or kNoCol
    int irw[NLD];           // (first) row within a pass
    int idst[NLD];          // LDS byte offset of the item's plane and columns
#pragma unroll
    for (int l = 0; l < NLD; ++l) {
        const int idx = tid + l * NT;
        const int h = idx % NH, cq = (idx / NH) % WCQ, img = (idx / NH / WCQ) % NI, rw = idx / NH / WCQ / NI * IR;
        irw[l] = rw;
        const int ic = ocol0 - g.PW + IC * cq;
        const bool any = (G8 || chof(h) < g.C) && rw < RWMAX;
        const uint32_t ioff = (uint32_t)img * (uint32_t)img_in + (uint32_t)chof(h);
#pragma unroll
        for (int k = 0; k < IC; ++k) icol[l][k] = any && ic + k >= 0 && ic + k < g.W ? (ioff + (uint32_t)((ic + k) * g.C)) * 2u : kNoCol;
        idst[l] = (img * CS + 8 * h) * CHP + 2 * IC * cq;
    }
    // the 2x2 average pool of x (MODE 2) leaves through a buffer descriptor as well: a store past its end is dropped
    __amdgpu_buffer_rsrc_t prsrc = xrsrc;
    if constexpr (POOL)
        prsrc = __builtin_amdgcn_make_buffer_rsrc(pool + (long long)b0 * g.AH * g.AW * g.C, (short)0,
                                                  (int)((long long)images * g.AH * g.AW * g.C * 2), 0x00020000);
    // Window row r of the run is stacked row orow0 - PH + r, counted from b0's first: where it lies (image group, row in it).
    // Rows between images and above the first are zeros; the host's `stack` keeps the windows of neighbouring images apart.
    const uint32_t row_in = (uint32_t)(g.W * g.C) * 2u, group_in = (uint32_t)img_in * (uint32_t)NI * 2u;
    auto locate = [&](int v, int& group, int& row) {
        group = images_in(max(v, 0)), row = v - group * g.per;   // (v < 0: row < 0)
    };
    // From pass 2 on a pass's 8 rows lie in two aligned groups of 8 stacked rows; images are a multiple of 8 rows apart, so a
    // group's place is uniform: row in the image and byte offset of groups a and b = a + 1, moved on by one each pass.
    const int row_w = orow0 - g.PH + 2 * RW01;   // (first row of pass 2)
    int ra, rb;
    uint32_t oa, ob;
    auto next_group = [&](int r, uint32_t o, int& rn, uint32_t& on) {
        const bool wrap = r + 8 >= g.per;
        rn = wrap ? 0 : r + 8, on = wrap ? o - (uint32_t)r * row_in + group_in : o + 8u * row_in;
    };
    {
        const int first = (row_w >> 3) * 8;   // (negative with paddings beyond the filter: rows above the image)
        const int group = images_in(max(first, 0));
        ra = first - group * g.per, oa = (uint32_t)group * group_in + (uint32_t)ra * row_in;
        next_group(ra, oa, rb, ob);
    }
    int lrow[NLD];          // the item's (first) row within its group
    bool inb[NLD];          // ... which is b
#pragma unroll
    for (int l = 0; l < NLD; ++l) {
        const int r = (row_w & 7) + irw[l];
        inb[l] = r >= 8, lrow[l] = irw[l] < 8 ? r & 7 : 0x40000000;   // (no item in these passes)
    }
    uint4 buf[2][NLD][IC * IR];
    auto load_item = [&](uint4 (&bf)[IC * IR], int l, bool ok, uint32_t off, bool ok1) {
#pragma unroll
        for (int r = 0; r < IR; ++r) {
            const uint32_t r0 = (r == 0 ? ok : ok1) ? off + (uint32_t)r * row_in : kNoRow;
#pragma unroll
            for (int k = 0; k < IC; ++k) bf[IC * r + k] = xload(r0 + icol[l][k]);
        }
    };
    auto issue_first = [&](uint4 (&bf)[NLD][IC * IR], int pass) {   // passes 0 and 1
#pragma unroll
        for (int l = 0; l < NLD; ++l) {
            int group, row;
            locate(orow0 - g.PH + pass * RW01 + irw[l], group, row);
            const bool ok = irw[l] < RW01;
            load_item(bf[l], l, ok && row >= 0 && row < g.H, (uint32_t)group * group_in + (uint32_t)row * row_in,
                      ok && row + 1 >= 0 && row + 1 < g.H);
        }
    };
    auto issue = [&](uint4 (&bf)[NLD][IC * IR], int pass) {   // passes from 2 on, in order; those past the window read nothing
        const bool any = first_row(pass) < NROWS;
        const int la = any && ra >= 0 ? g.H - ra : 0, lb = any && rb >= 0 ? g.H - rb : 0;
#pragma unroll
        for (int l = 0; l < NLD; ++l) {
            const int lim = inb[l] ? lb : la;
            load_item(bf[l], l, lrow[l] < lim, (inb[l] ? ob : oa) + (uint32_t)(lrow[l] & 7) * row_in, lrow[l] + 1 < lim);
        }
        ra = rb, oa = ob;
        next_group(rb, ob, rb, ob);
    };
    // A pass into the window: the columns of channels 2j and 2j + 1 of the items' rows at ring byte offset cring[l].  No
    // branch, so that the products around it can be interleaved: lanes without an item write to spare bytes (with FEW
    // products there is nothing to interleave, and wavefronts without an item write nothing).
    int cring[NLD];
    constexpr int ITEMS = RWMAX / IR * NI * WCQ * NH;
    const int wave0 = __builtin_amdgcn_readfirstlane(tid) & ~63;   // the wavefront's first thread
    auto commit_part = [&](const uint4 (&bf)[NLD][IC * IR], int j) {
#pragma unroll
        for (int l = 0; l < NLD; ++l) {
            if (FEW && wave0 + l * NT >= ITEMS) continue;   // (uniform)
#pragma unroll
            for (int r = 0; r < IR; ++r) {
                auto d = [&](int k) { const uint4& u = bf[l][IC * r + k]; return j == 0 ? u.x : j == 1 ? u.y : j == 2 ? u.z : u.w; };
                char* const dst = xl + cring[l] + r * RP;   // (a pair of rows never wraps: both even)
#pragma unroll
                for (int odd = 0; odd < 2; ++odd) {
                    const uint32_t sel = odd ? 0x07060302u : 0x05040100u;
                    const uint32_t lo = __builtin_amdgcn_perm(d(1), d(0), sel);
                    if constexpr (IC == 4)
                        *reinterpret_cast<uint2*>(dst + (2 * j + odd) * CHP) = make_uint2(lo, __builtin_amdgcn_perm(d(3), d(2), sel));
                    else
                        *reinterpret_cast<uint32_t*>(dst + (2 * j + odd) * CHP) = lo;
                }
            }
        }
    };
    auto commit_next = [&]() {   // 8 rows on (passes from 2 on)
#pragma unroll
        for (int l = 0; l < NLD; ++l) {
            cring[l] += irw[l] < 8 ? 8 * RP : 0;
            cring[l] -= irw[l] < 8 && cring[l] - idst[l] >= NRR * RP ? NRR * RP : 0;
        }
    };
    auto write_pool = [&](const uint4 (&bf)[NLD][IC * IR], int pass) {
        if constexpr (POOL) {
            const int wr0 = first_row(pass), nrw = pass < 2 ? RW01 : 8;
#pragma unroll
            for (int l = 0; l < NLD; ++l) {
                // the thread holds one window of the 2x2 pool (H, W, PH, PW even): the run that owns these rows writes it
                const int idx = tid + l * NT;
                const int h = idx % NH, cq = (idx / NH) % WCQ, img = (idx / NH / WCQ) % NI;
                const int v = orow0 - g.PH + wr0 + irw[l], ic = ocol0 - g.PW + 2 * cq;
                int group, ir;
                locate(v, group, ir);
                const bool mine = irw[l] < nrw && chof(h) < g.C && v >= orow0 && v < orow0 + rows_valid && ir < g.H &&
                                  ic >= ocol0 && ic < ocol0 + cols_valid;
                union U {
                    uint4 u;
                    T t[8];
                } p0, p1, p2, p3, o;
                p0.u = bf[l][0], p1.u = bf[l][1], p2.u = bf[l][2], p3.u = bf[l][3];
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    o.t[e] = from_f32<T>((((to_f32(p0.t[e]) + to_f32(p1.t[e])) + to_f32(p2.t[e])) + to_f32(p3.t[e])) * 0.25f);
                const uint32_t off = mine ? (uint32_t)((((group * NI + img) * g.AH + (ir >> 1)) * g.AW + (ic >> 1)) * g.C + chof(h)) * 2u : kNoRow;
                typedef unsigned v4u __attribute__((ext_vector_type(4)));
                __builtin_amdgcn_raw_buffer_store_b128(v4u{o.u.x, o.u.y, o.u.z, o.u.w}, prsrc, (int)off, 0, 0);
            }
        }
    };
    auto commit_first = [&](const uint4 (&bf)[NLD][IC * IR], int pass) {   // passes 0 and 1
#pragma unroll
        for (int l = 0; l < NLD; ++l) cring[l] = irw[l] < RW01 ? idst[l] + (pass * RW01 + irw[l]) % NRR * RP : Sh::spare(POOL);
#pragma unroll
        for (int j = 0; j < 4; ++j) commit_part(bf, j);
        write_pool(bf, pass);
    };
    issue_first(buf[0], 0);
    issue_first(buf[1], 1);

    // LDS accesses of this wavefront complete, then the workgroup barrier; global loads and stores stay in flight
    auto lds_barrier = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    // ---- filter table wt[copy][channel][3 + u][3 + v] (rotated for the input gradient), zero elsewhere; copy 1 is
    // the same table one element to the left, so that a run of 8 values that starts at an odd index is dword
    // aligned in it
    constexpr int WTC = CS * WTH * WTW;  // elements per copy
    unsigned short* const wt = reinterpret_cast<unsigned short*>(r2);
    {
        uint4* wz = reinterpret_cast<uint4*>(r2);
        for (int i = tid; i < (2 * Sh::WTB + 15) / 16; i += NT) wz[i] = make_uint4(0u, 0u, 0u, 0u);
        lds_barrier();
#pragma unroll
        for (int i = 0; i < NWL; ++i) {
            const int idx = tid + i * NT;
            const int h = idx % NH, uv = idx / NH;
            const int u = uv / K, v = uv - u * K;
            if (idx < K * K * NH && (G8 || chof(h) < g.C)) {
                const uint32_t d[4] = {wval[i].x, wval[i].y, wval[i].z, wval[i].w};
                const int uu = g.flip ? K - 1 - u : u, vv = g.flip ? K - 1 - v : v;
                unsigned short* wp = wt + ((8 * h) * WTH + 3 + uu) * WTW + 3 + vv;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const unsigned short val = (unsigned short)((d[e >> 1] >> (16 * (e & 1))) & 0xffffu);
                    wp[e * WTH * WTW] = val;
                    wp[WTC + e * WTH * WTW - 1] = val;
                }
            }
        }
        // (the table is read after the barrier that also publishes the window's first passes)
    }
    const int ln = lane & 15, kg = lane >> 4;
    // ---- per-lane addresses
    // B operands: lane = (patch n = image * NPC + pc, k group kg); operand a = ICB * rowgroup + i covers window rows
    // 4 rowgroup + (4i + kg) / ICB, column block (4i + kg) % ICB
    const int pimg = ln / NPC, pc = ln % NPC;
    const char* xb[CPW][ICB];
#pragma unroll
    for (int q = 0; q < CPW; ++q)
#pragma unroll
        for (int i = 0; i < ICB; ++i)
            xb[q][i] = xl + (pimg * CS + wv * CPW + q) * CHP + ((4 * i + kg) / ICB) * RP + ((4 * i + kg) % ICB) * 16 + pc * 8;
    // results: register r of a lane is output (row kg, column 4 pc + r) of patch n
    char* const olw = r2 + (pimg * 4 + kg) * OROWP + (4 * pc) * OPX + pc * 4 + 2 * (wv * CPW);
    // store phase: one 16-byte piece (image, row, column, h) of each 4-row result tile per thread, through buffer
    // descriptors (an offset past the end: nothing stored / zero loaded), so that no vector memory instruction of the
    // kernel sits behind a branch and the in-flight counts the staging waits rely on stay exact
    const int sh = tid % NH, scol = (tid / NH) % TW, srow = (tid / NH / TW) % 4, simg = tid / NH / TW / 4 % NI;
    const int stile = tid / Sh::PIECES;   // (with TPT = 2: the tile of the step's two that the thread stores)
    auto tile_of = [&](int n) { return Sh::TPT == 2 ? stile : n; };
    const bool s_ok = stile < Sh::TPT && scol < cols_valid && (GATE || c0 + 8 * sh < g.C);
    const char* const olr = r2 + (simg * 4 + srow) * OROWP + scol * OPX + (scol >> 2) * 4 + 16 * sh;
    const __amdgpu_buffer_rsrc_t yrsrc = __builtin_amdgcn_make_buffer_rsrc(
        y + (long long)b0 * img_out, (short)0, (int)(images * img_out * 2), 0x00020000);
    const uint32_t ycol = (uint32_t)simg * (uint32_t)img_out +
                          (uint32_t)((ocol0 + scol) * g.YC + g.ych + (G8 ? 4 * sl : GATE ? 8 * sl + 4 * sh : c0 + 8 * sh));
    __amdgpu_buffer_rsrc_t arsrc = xrsrc;
    if constexpr (ADD)
        arsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(add + (long long)b0 * g.AH * g.AW * g.C), (short)0,
                                                  (int)((long long)images * g.AH * g.AW * g.C * 2), 0x00020000);
    constexpr int NA = ANY ? 4 : 1;   // addends of a piece
    uint4 addv[NG][NA];
    // ANY: the bins of an image's rows in LDS, as the byte offset of the first and bits: it is the longer of the two lengths that bins have, there is
    // a second, that is the longer.  A bin's weight is one over its pixels, for a thread's column one of two by the row's bin (a product of one
    // over each length is 7e-8 off for 3 x 3 pixels, where that is exact to 1e-8).
    uint2* const bins = reinterpret_cast<uint2*>(xl + Sh::bins_at);
    int jb0 = 0;
    float wj[2][2] = {};   // [the row's bin is the longer][the column's first or second bin; 0: not there]
    uint32_t wi[NG] = {};
    if constexpr (ANY) {
        const int least = (g.OH + g.AH - 1) / g.AH;
        for (int i = tid; i < g.OH; i += NT) {   // (read behind the barrier that publishes the first passes)
            int b, l0, l1;
            pool_bin_lengths(i, g.OH, g.AH, b, l0, l1);
            bins[i] = make_uint2((uint32_t)(b * g.AW * g.C) * 2u, (l0 > least ? 1u : 0u) | (l1 > 0 ? 2u : 0u) | (l1 > least ? 4u : 0u));
        }
        int l0, l1;
        pool_bin_lengths(min(ocol0 + scol, g.OW - 1), g.OW, g.AW, jb0, l0, l1);
#pragma unroll
        for (int p = 0; p < 2; ++p) wj[p][0] = 1.f / (float)((least + p) * l0), wj[p][1] = l1 > 0 ? 1.f / (float)((least + p) * l1) : 0.f;
    }
    // a step's 8 rows lie in one image (group): its first row there, and the byte offsets of that row in y and the addend
    int orow = orow0, rleft = rows_valid;   // rleft: rows of the run from this step on
    const uint32_t row_out = (uint32_t)(g.OW * g.YC) * 2u, group_out = (uint32_t)img_out * (uint32_t)NI * 2u;
    const uint32_t row_add = (uint32_t)(g.AW * g.C) * 2u, group_add = (uint32_t)(NI * g.AH) * row_add;
    uint32_t ooff = (uint32_t)orow * row_out, aoff = ANY ? 0u : (uint32_t)(orow >> 1) * row_add, stored = 0;   // stored: ooff of the step before
    uint32_t ylane[NG], alane[NG], yoff[NG];   // the thread's piece from there (rows srow or srow + 4); yoff: or the marker
#pragma unroll
    for (int n = 0; n < NG; ++n) {
        const int r = 4 * tile_of(n) + srow;
        ylane[n] = s_ok ? ycol * 2u + (uint32_t)r * row_out : kNoRow;
        if constexpr (ANY) alane[n] = (uint32_t)((simg * g.AH * g.AW + jb0) * g.C + c0 + 8 * sh) * 2u;
        else alane[n] = s_ok ? (uint32_t)(((simg * g.AH + (r >> 1)) * g.AW + ((ocol0 + scol) >> 1)) * g.C + c0 + 8 * sh) * 2u : kNoRow;
        yoff[n] = kNoRow;
#pragma unroll
        for (int t = 0; t < NA; ++t) addv[n][t] = make_uint4(0u, 0u, 0u, 0u);
    }
    // The next step: the offsets its tiles are stored at, and the addends.  (A step between images moves nothing and takes no scalar
    // offset: behind images of one to three rows it could lie past the descriptor's end, from which the range check subtracts it.)
    auto place = [&]() {
        const int lim = min(g.OH - orow, rleft);
#pragma unroll
        for (int n = 0; n < NG; ++n) {
            const bool ok = 4 * tile_of(n) + srow < lim;
            yoff[n] = ok ? ylane[n] : kNoRow;
            if constexpr (ANY) {
                const bool in = ok && s_ok;
                const uint2 bin = bins[ok ? orow + 4 * tile_of(n) + srow : 0];
                const uint32_t o = alane[n] + bin.x;
                wi[n] = bin.y;
                const bool right = in && wj[0][1] != 0.f, below = in && (bin.y & 2u) != 0;
                const uint32_t at = lim > 0 ? aoff : 0;
                addv[n][0] = xload_from(arsrc, in ? o : kNoRow, at);
                addv[n][1] = xload_from(arsrc, right ? o + 2u * (uint32_t)g.C : kNoRow, at);
                addv[n][2] = xload_from(arsrc, below ? o + row_add : kNoRow, at);
                addv[n][3] = xload_from(arsrc, right && below ? o + row_add + 2u * (uint32_t)g.C : kNoRow, at);
            } else if constexpr (ADD) {
                addv[n][0] = xload_from(arsrc, ok ? alane[n] : kNoRow, lim > 0 ? aoff : 0);
            }
        }
        stored = lim > 0 ? ooff : 0;
        rleft -= 8, orow += 8;
        const bool wrap = orow >= g.per;
        ooff += wrap ? group_out - (uint32_t)(orow - 8) * row_out : 8u * row_out;
        aoff += ANY ? (wrap ? group_add : 0u) : wrap ? group_add - (uint32_t)((orow - 8) >> 1) * row_add : 4u * row_add;
        orow = wrap ? 0 : orow;
    };
    auto tile_read = [&](int f, int n) {
        const char* src = olr + (2 * (f & 1) + min(tile_of(n), 1)) * OLB;   // (f: or anything of its parity)
        if constexpr (GATE) {
            // the thread gates 4 channel pairs of the pixel: values 4 sh .. 4 sh + 3 of both 8-channel pieces, or
            // the two halves of an 8-channel slice's one piece
            const char* sg = G8 ? src : src - 8 * sh;   // (src points 16 sh into the pixel)
            constexpr int PB = G8 ? 8 : 16;             // bytes between a pair's two values
            return make_uint4(*reinterpret_cast<const uint32_t*>(sg), *reinterpret_cast<const uint32_t*>(sg + 4),
                              *reinterpret_cast<const uint32_t*>(sg + PB), *reinterpret_cast<const uint32_t*>(sg + PB + 4));
        } else {
            return make_uint4(*reinterpret_cast<const uint32_t*>(src), *reinterpret_cast<const uint32_t*>(src + 4),
                              *reinterpret_cast<const uint32_t*>(src + 8), *reinterpret_cast<const uint32_t*>(src + 12));
        }
    };
    auto tile_store = [&](uint4 v, int n) {   // where place() put it
        if constexpr (ANY) {
            const bool top = (wi[n] & 1u) != 0, below = (wi[n] & 4u) != 0;
            v = tz_add_bins<T>(v, addv[n], top ? wj[1][0] : wj[0][0], top ? wj[1][1] : wj[0][1], below ? wj[1][0] : wj[0][0], below ? wj[1][1] : wj[0][1]);
        } else if constexpr (ADD) v = tz_add_quarter<T>(v, addv[n][0]);
        if constexpr (GATE) {
            const uint2 o = tz_gate<T>(make_uint2(v.x, v.y), make_uint2(v.z, v.w), g.gs);
            typedef unsigned v2u __attribute__((ext_vector_type(2)));
            __builtin_amdgcn_raw_buffer_store_b64(v2u{o.x, o.y}, yrsrc, (int)yoff[n], (int)stored, 0);
        } else {
            typedef unsigned v4u __attribute__((ext_vector_type(4)));
            // (No scalar offset in a 16-byte store: with one the compiler leaves no wait state between the store and a vector
            // instruction that overwrites its data registers, and the last quarter of a row of lanes then stores the new value.)
            __builtin_amdgcn_raw_buffer_store_b128(v4u{v.x, v.y, v.z, v.w}, yrsrc, (int)(yoff[n] + stored), 0, 0);
        }
    };

    uint4 ring[CPW][RING];
    auto read16 = [&](const char* p) {
        const uint2 lo = *reinterpret_cast<const uint2*>(p), hi = *reinterpret_cast<const uint2*>(p + 8);
        return make_uint4(lo.x, lo.y, hi.x, hi.y);
    };
    auto load_group = [&](int slotgroup, int byteoff) {  // window rows byteoff / RP .. + 3 -> ICB operands per channel
#pragma unroll
        for (int q = 0; q < CPW; ++q)
#pragma unroll
            for (int i = 0; i < ICB; ++i) ring[q][slotgroup * ICB + i] = read16(xb[q][i] + byteoff);
    };
    // the passes the first step reads, then the ring's first PER - 1 row groups
    commit_first(buf[0], 0);
    if constexpr (PASSES > 2) issue(buf[0], 2);
    commit_first(buf[1], 1);
    if constexpr (PASSES > 3) issue(buf[1], 3);
#pragma unroll
    for (int l = 0; l < NLD; ++l) cring[l] = irw[l] < 8 ? idst[l] + (2 * RW01 + irw[l]) % NRR * RP : Sh::spare(POOL);
    lds_barrier();
    // ---- this wavefront's A operands: lane = (m = 4 di + dj, k group kg); operand t covers k groups 4t .. 4t+3
    uint4 A[CPW][NM];
    {
        const int di = ln >> 2, dj = ln & 3;
#pragma unroll
        for (int q = 0; q < CPW; ++q) {
#pragma unroll
            for (int t = 0; t < NM; ++t) {
                const int kap = 4 * t + kg;
                const int r = kap / ICB, cb = kap - r * ICB;
                const int v0 = 8 * cb - dj + 3;  // first of the lane's 8 table columns
                const uint32_t* wp = reinterpret_cast<const uint32_t*>(
                    wt + (v0 & 1) * WTC + ((wv * CPW + q) * WTH + r - di + 3) * WTW + (v0 & ~1));
                const bool real = kap < NKG;
                A[q][t] = make_uint4(real ? wp[0] : 0u, real ? wp[1] : 0u, real ? wp[2] : 0u, real ? wp[3] : 0u);
            }
        }
    }

#pragma unroll
    for (int j = 0; j < PER - 1; ++j) load_group(j, 4 * j * RP);
    // A step is two row groups (8 output rows), UNRF steps (the ring's period in steps) a trip.
    const int nfat = (nsteps + 1) >> 1;
    // (commits: a step follows; issues: passes from f + 4 on may lie in the window)
    auto step = [&](int jf, int f, auto commits, auto issues) __attribute__((always_inline)) {
        constexpr bool COMMITS = decltype(commits)::value, ISSUES = decltype(issues)::value;
        // the two row groups this step adds to the ring; the second goes to the slot of the step's own first group, once the
        // first tile's products with that are issued (LATE), or waits in registers where those are nearly all there are
        constexpr bool LATE = PER >= 3;
        uint4 out[NG];
        auto tiles_read = [&]() {
#pragma unroll
            for (int n = 0; n < NG; ++n) out[n] = tile_read(jf + 1, n);
        };
        auto tiles_store = [&]() {
#pragma unroll
            for (int n = 0; n < NG; ++n) tile_store(out[n], n);
        };
        if constexpr (FEW) {
            tiles_read();
            __builtin_amdgcn_sched_barrier(0x6);
        }
        load_group((2 * jf + PER - 1) % PER, ((2 * f + PER - 1) % NR) * (4 * RP));
        const int late_off = ((2 * f + PER) % NR) * (4 * RP);
        uint4 late[CPW][ICB];
        if constexpr (!LATE) {
#pragma unroll
            for (int q = 0; q < CPW; ++q)
#pragma unroll
                for (int i = 0; i < ICB; ++i) late[q][i] = read16(xb[q][i] + late_off);
        }
        if constexpr (FEW) {
            __builtin_amdgcn_sched_barrier(0x6);
            tiles_store();
            __builtin_amdgcn_sched_barrier(0x6);
        } else {
            tiles_read();
        }
        tz_f32x4 acc[2][CPW];
#pragma unroll
        for (int gi = 0; gi < 2; ++gi)
#pragma unroll
            for (int q = 0; q < CPW; ++q) acc[gi][q] = tz_f32x4{0.f, 0.f, 0.f, 0.f};
        // The products, and between them what moves data: the previous step's tiles out, the pass the NEXT step needs into
        // the window, the one two steps on requested.  (One after the other they leave the matrix pipe idle two thirds of
        // a step; left to itself the compiler puts them one after the other.)
        constexpr int MOVE = NM < 7 ? 1 : NM / 7;   // products per channel and tile between two pieces
#pragma unroll
        for (int t = 0; t < NM; ++t) {
#pragma unroll
            for (int q = 0; q < CPW; ++q) {
                acc[0][q] = mfma16(A[q][t], ring[q][(ICB * 2 * jf + t) % RING], acc[0][q], T());
                const uint4 b1 = LATE || t < ICB * (PER - 1) ? ring[q][(ICB * (2 * jf + 1) + t) % RING] : late[q][t - ICB * (PER - 1) < ICB ? t - ICB * (PER - 1) : 0];
                acc[1][q] = mfma16(A[q][t], b1, acc[1][q], T());
            }
            if constexpr (LATE) {
                if (t == ICB - 1) load_group((2 * jf) % PER, late_off);
            }
#pragma unroll
            for (int piece = 0; piece < 7; ++piece) {
                if (t != (piece * MOVE < NM - 1 ? piece * MOVE : NM - 1)) continue;
                if (COMMITS && piece >= 2 && piece < 6) commit_part(buf[jf % 2], piece - 2);   // pass f + 2 sits in buffer f % 2 = jf % 2 (UNRF is even)
                if (COMMITS && piece == 6) {
                    commit_next();
                    write_pool(buf[jf % 2], f + 2);
                    if constexpr (ISSUES) issue(buf[jf % 2], f + 4);
                }
                if (piece == 0 && !FEW) tiles_store();
                if (piece == 1) place();
                __builtin_amdgcn_sched_barrier(0x6);   // (vector and scalar arithmetic may cross)
            }
        }
        if constexpr (!LATE) {
#pragma unroll
            for (int q = 0; q < CPW; ++q)
#pragma unroll
                for (int i = 0; i < ICB; ++i) ring[q][((2 * jf) % PER) * ICB + i] = late[q][i];
        }
#pragma unroll
        for (int gi = 0; gi < 2; ++gi) {
            char* dst = olw + (2 * (jf & 1) + gi) * OLB;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if constexpr (CPW == 2) {
                    union {
                        T t[2];
                        uint32_t u;
                    } o;
                    o.t[0] = from_f32<T>(acc[gi][0][r]), o.t[1] = from_f32<T>(acc[gi][1][r]);
                    *reinterpret_cast<uint32_t*>(dst + r * OPX) = o.u;
                } else {
                    *reinterpret_cast<T*>(dst + r * OPX) = from_f32<T>(acc[gi][0][r]);
                }
            }
        }
    };
    constexpr std::true_type yes;
    constexpr std::false_type no;
    auto any = [&](int jf, int f, auto commits, auto issues) __attribute__((always_inline)) {
        lds_barrier();  // the previous step's tiles are complete, its window reads done
        step(jf, f, commits, issues);
    };
    int last = 0;   // (the parity known where it is set: 188 registers at filter 17, 231 with nfat - 1)
    if constexpr (SHORT == 2) {
        if (nfat == 2) any(0, 0, yes, no), any(1, 1, no, no), last = 1;   // (uniform)
        else any(0, 0, no, no);
    } else if constexpr (SHORT == 1) {
        any(0, 0, no, no);
    } else if constexpr (UNRF <= 6) {
        // Whole trips, then what is left of the run by itself: with a way out between the steps of a trip the compiler no longer
        // knows which requests are the newest, and commits waited for those of the step before as well (us: [32,56,56,128] filter 13
        // 17.0 -> 16.6, 9 15.5 -> 15.0, 7 15.3 -> 14.8; [16,32,32,64] 7.25 -> 6.9, 6.6 -> 6.3, 6.4 -> 6.15).  In turn and not by the
        // compiler's unrolling, which gives up on a loop with so many ways out.
        int f0 = 0;
        auto trip = [&](auto jf) { return any(jf, f0 + jf, yes, yes), last = f0 + jf, true; };
        auto left = [&](auto jf) { return f0 + jf < nfat && trip(jf); };   // (uniform)
        for (; f0 + UNRF <= nfat; f0 += UNRF) tz_in_turn<0, UNRF>(trip);
        tz_in_turn<0, UNRF - 1>(left);
    } else {
        // Ten steps a trip, left after the run's last step: few runs take a second one, and nine more steps of code cost more than
        // the waits (us, [32,56,56,128] filter 17 25.6 and 25.8, [32,28,28,64] 9.15 and 9.35).
        bool left = false;
        for (int f0 = 0; f0 < nfat; f0 += UNRF) {
#pragma unroll
            for (int jf = 0; jf < UNRF; ++jf) {
                any(jf, f0 + jf, yes, yes);
                if (f0 + jf + 1 >= nfat) {   // (uniform)
                    left = true, last = f0 + jf;
                    break;
                }
            }
            if (left) break;
            last = f0 + UNRF - 1;
        }
    }
    lds_barrier();
#pragma unroll
    for (int n = 0; n < NG; ++n) tile_store(tile_read(last, n), n);
}

template <typename T, int K, int NPC, int CS, int MODE>
__global__ __launch_bounds__(512, 1) void dwconv_tz_k(const T* __restrict__ x, const T* __restrict__ w,
                                                      const T* __restrict__ add, T* __restrict__ pool,
                                                      T* __restrict__ y, const TzGeom g) {
    dwconv_tz_body<T, K, NPC, CS, MODE>(x, w, add, pool, y, g, blockIdx.x, gridDim.x);
}

// ------------------------------------------------------------------------------------------------
// Host side

// Patches per image row, 16 (true) or 8 in two images: the width whose padding of (columns x images) is smaller, wider on ties.
inline bool tz_wide_tile(int B, int OW) {
    return (long long)cdiv(OW, 64) * 64 * B <= (long long)cdiv(OW, 32) * 32 * cdiv(B, 2) * 2;
}

// Rows of the stack (of one image where there is none).
inline int tz_rows(const TzGeom& g, int ni) { return g.stack ? (cdiv(g.B, ni) - 1) * g.stack + g.OH : g.OH; }

// Cuts the stack into runs of `run` rows (a multiple of 8), or every image by itself where that makes no more of them (its last
// run may be shorter, and none needs the rows between two images) or there is no stack; false: a run's images are beyond 32-bit
// offsets.  (us, by the image only where the run divided the image's rows of the stack, and now: [32,28,28,64] filter 17 9.4 -> 8.5,
// 15 9.4 -> 8.55; both scales of [8,112,112,48], filter 17, 16.1 -> 15.2; elsewhere the same.)
inline bool tz_cut(TzGeom& g, int ni, long long run) {
    const int images = cdiv(g.B, ni), total = tz_rows(g, ni);
    if (run > total) run = (total + 7) / 8 * 8;
    g.run = (int)run, g.rpi = cdiv(g.OH, g.run);
    const long long alone = (long long)images * g.rpi;
    if (g.stack && alone > cdiv(total, g.run)) g.rpi = 0;
    if (g.rpi && alone > 0x7fffffffLL) return false;
    g.nruns = g.rpi ? (int)alone : cdiv(total, g.run);
    const long long reach = g.rpi ? ni : ((long long)(g.stack + g.run + 64) / g.stack + 1) * ni, most = reach < g.B ? reach : g.B;
    const long long in = (long long)g.H * g.W * g.C, out = (long long)g.OH * g.OW * g.YC;
    // the kernel's quotients of workgroups: by slices, tiles and runs
    const int by = std::max(std::max(g.nslices, g.ncolt), g.rpi);
    if ((long long)g.nruns * g.ncolt * g.nslices * by > 0xffffffffLL) return false;
    g.per = g.rpi ? kTzAlone : g.stack, g.per_inv = g.rpi ? kTzAloneInverse : tz_inverse(g.stack), g.rpi_inv = tz_inverse(std::max(g.rpi, 1));
    g.ncolt_inv = tz_inverse(g.ncolt), g.nslices_inv = tz_inverse(g.nslices);
    return most * (in > out ? in : out) <= 0x1fffffffLL;
}
inline long long tz_blocks(const TzGeom& g) { return (long long)g.nruns * g.ncolt * g.nslices; }

// Steps of 8 rows of the longest run: those between images at a run's end are left out.
inline int tz_steps(const TzGeom& g) {
    if (g.rpi) return (std::min(g.run, g.OH) + 7) / 8;
    return (g.run % g.stack == 0 ? g.run - g.stack + g.OH + 7 : g.run) / 8;
}

// Price of a workgroup to the planners of shared launches, us: a start-up (first windows, filter table, operand set-up), then steps of
// 8 rows.  (The step is that of runs which have the memory to themselves.  256 equal runs at once take 6.1 + 1.47 a step at
// [64,H,56,64] filter 13, 5.5 + 1.36 at filter 9, 5.9 + 1.2 at filter 15 with its 8 channels; with the pooled gradient 6.1 + 1.8, 5.7 +
// 1.6 and 6.1 + 1.35.)
constexpr double kTzStart = 7.0, kTzStep = 0.9;

// The cut with the fewest workgroups whose runs have at most `steps` steps (of equal ones the shorter runs): runs of any length,
// whole images, or equal parts of an image.
inline bool tz_cut_steps(TzGeom& g, int ni, int steps) {
    long long best = 0, best_blocks = 0;
    int best_steps = 0;
    auto look = [&](long long run) {
        if (run < 8 || !tz_cut(g, ni, run) || tz_steps(g) > steps) return;
        const long long n = tz_blocks(g);
        if (best == 0 || n < best_blocks || (n == best_blocks && tz_steps(g) < best_steps)) best = run, best_blocks = n, best_steps = tz_steps(g);
    };
    const int per_image = cdiv(g.OH, 8);
    look(8LL * steps);
    if (steps < per_image) {
        look(8LL * cdiv(per_image, cdiv(per_image, steps)));
    } else {
        const long long n = g.stack ? (steps - per_image) / (g.stack / 8) + 1 : 1;
        look(n == 1 ? 8LL * per_image : n * g.stack);
    }
    return best != 0 && tz_cut(g, ni, best);
}

// Time of a launch of equal runs by itself, in steps of one that has its compute unit to itself, to its planner: what a unit takes of
// them, one after the other, each with a start-up of 4.5 (of 5 it tied 18 steps in 435 workgroups with 10 in 696 at [16,81,78,232]
// filter 17: 64 and 54 us; what 256 equal runs at once take says 4.0 to 4.9); with `pairs` (filters 3 and 5) a unit holds two, which take less than twice as long
// (us, [1725,8,9,56] filter 3: 27 steps in 256 workgroups 26.5, 13 in 496 22.9, 9 in 768 25.0).
inline double tz_alone_cost(long long blocks, int steps, bool pairs) {
    if (!pairs) return (double)cdiv(blocks, 256) * (4.5 + steps);
    return blocks <= 256 ? 5.0 + steps : 7.5 + 0.8 * steps * cdiv(blocks, 256) + 2.5 * (cdiv(blocks, 512) - 1);
}

// Runs of a launch of its own: the cut estimated to end first of those that fill 256 compute units 1..8 times, the equal parts of
// an image and numbers of whole images; false: not covered.  (480 random shapes with all of about 20 cuts timed: the choice is 0.2 %
// behind the fastest, 0.6 % at filters 3 and 5; at a price of eight steps a start-up, four fillings, and parts or whole images only next
// to those it was 3 %, 38 % at worst.  us: [16,77,76,232] filter 15 62.8 -> 51, 5 28.9 -> 24.8, [144,8,7,1112] filter 3 43.1 -> 33.)
inline bool tz_cut_alone(TzGeom& g, int ni, bool pairs = false) {
    const long long per_run = (long long)g.ncolt * g.nslices;
    const int images = cdiv(g.B, ni), per_image = cdiv(g.OH, 8);
    const long long total = cdiv(tz_rows(g, ni), 8) * (g.stack ? 1LL : images);
    long long best = 0;
    double best_cost = 0;
    auto look = [&](long long run) {
        if (!tz_cut(g, ni, run)) return;
        const double cost = tz_alone_cost(tz_blocks(g), tz_steps(g), pairs);
        if (best == 0 || cost < best_cost) best = run, best_cost = cost;
    };
    for (int rounds = 1; rounds <= 8; ++rounds) {
        const long long want = 256LL * rounds / per_run, n = want < 1 ? 1 : want > total ? total : want;
        look(8LL * cdiv(total, n));
    }
    for (int parts = 1; parts <= std::min(per_image, 16); ++parts) look(8LL * cdiv(per_image, parts));
    if (g.stack)
        for (int n = 1; n <= std::min(images, 16); ++n) look((long long)n * g.stack);
    // (large images: runs as short as their offsets need)
    return tz_cut(g, ni, best == 0 ? 8 : best) && tz_blocks(g) <= 0x7fffffffLL;
}

// The geometry but for the runs (false: not covered).
template <int K, int NPC, int CS>
static bool tz_make_geom(TzGeom& g, bool add, int B, int H, int W, int C, int PH, int PW, bool flip, const TzGate* gate) {
    using Sh = TzShape<K, NPC, CS>;
    g.B = B, g.H = H, g.W = W, g.C = C, g.PH = PH, g.PW = PW, g.flip = flip ? 1 : 0;
    g.OH = H + 2 * PH - K + 1, g.OW = W + 2 * PW - K + 1;
    g.AH = add ? g.OH / 2 : H / 2, g.AW = add ? g.OW / 2 : W / 2;
    g.YC = gate ? gate->ldy : C, g.ych = gate ? gate->ych : 0, g.gs = gate ? gate->gs : 1.f;
    if (gate && (add || flip || C % 16 != 0 || gate->ldy < gate->ych + C / 2 || (gate->ldy | gate->ych) % 8 != 0)) return false;
    if ((long long)H * W * C * Sh::NI > 0x1fffffffLL || (long long)g.OH * g.OW * g.YC * Sh::NI > 0x1fffffffLL) return false;
    // the windows of an image's first patches reach PH rows above it, and the operands of its last, output rows 4 * ((OH - 1) / 4)
    // on, OPR rows from PH above those: none of them the neighbour's
    g.stack = (std::max(std::max(H + PH, g.OH), 4 * ((g.OH - 1) / 4) - PH + Sh::OPR) + 7) / 8 * 8;
    // the kernel's quotients of rows of the stack by this are exact up to 2^32 / stack; images too tall for that are walked one by
    // one (a run of one such image is thousands of steps: nothing is lost)
    const long long rows = (long long)cdiv(B, Sh::NI) * g.stack;
    if (rows > 0x3fffffffLL || (2 * rows + g.stack + 128) * g.stack > 0xffffffffLL) g.stack = 0;
    g.ncolt = cdiv(g.OW, Sh::TW), g.nslices = cdiv(C, CS);
    return true;
}

template <typename T, int K, int NPC, int CS>
static int launch_tz(const void* x, const void* w, const void* add, void* pool, void* y, int B, int H, int W, int C,
                     int PH, int PW, bool flip, const TzGate* gate, hipStream_t s) {
    using Sh = TzShape<K, NPC, CS>;
    TzGeom g;
    if (!tz_make_geom<K, NPC, CS>(g, add != nullptr, B, H, W, C, PH, PW, flip, gate)) return -1;
    // (the search takes 0.66 us of the call, which a short kernel does not hide; kept 0.02)
    const bool pairs = K <= 5 && !pool;
    static PlanCache<std::array<int, 8>, TzRuns> plans;
    static_cast<TzRuns&>(g) = plans.get({B, H, W, C, PH, PW, g.YC, pairs}, [=]() mutable {
        if (!tz_cut_alone(g, Sh::NI, pairs)) g.nruns = 0;
        return static_cast<TzRuns>(g);
    });
    if (g.nruns == 0) return -1;
    const size_t lds = pool ? Sh::lds_bytes_pool : Sh::lds_bytes;
    const bool brief = !pool && tz_steps(g) <= tz_short(K);
    const int mode = (add ? 1 : 0) | (pool ? 2 : 0) | (gate ? 4 : 0) | (brief ? 8 : 0);
    auto kern = dwconv_tz_k<T, K, NPC, CS, 0>;
    if (mode == 1) kern = dwconv_tz_k<T, K, NPC, CS, 1>;
    if (mode == 2) kern = dwconv_tz_k<T, K, NPC, CS, 2>;
    if (mode == 4) kern = dwconv_tz_k<T, K, NPC, CS, 4>;
    if constexpr (CS == 16) {
        if (mode == 6) kern = dwconv_tz_k<T, K, NPC, CS, 6>;
    }
    if constexpr (tz_short(K) != 0) {
        if (mode == 8) kern = dwconv_tz_k<T, K, NPC, CS, 8>;
        if (mode == 9) kern = dwconv_tz_k<T, K, NPC, CS, 9>;
        if (mode == 12) kern = dwconv_tz_k<T, K, NPC, CS, 12>;
    }
    if ((mode & 7) == 3 || (mode & 7) == 5 || (mode & 7) == 7 || (mode == 6 && CS != 16)) return -1;
    static std::once_flag attr_once[16];
    std::call_once(attr_once[mode], [&] { (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); });
    hipLaunchKernelGGL(kern, dim3((unsigned)tz_blocks(g)), dim3(Sh::NT), lds, s, (const T*)x, (const T*)w, (const T*)add,
                       (T*)pool, (T*)y, g);
    return check_launch("dwconv_tz");
}

// -1: not covered (the caller falls back to the other kernels).
template <typename T, int K>
static int launch_tz_best(const void* x, const void* w, const void* add, void* pool, void* y, int B, int H, int W, int C,
                          int PH, int PW, bool flip, const TzGate* gate, hipStream_t s) {
    const int OH = H + 2 * PH - K + 1, OW = W + 2 * PW - K + 1;
    if (OH < 1 || OW < 1 || C % 8 != 0 || B < 1) return -1;
    if ((reinterpret_cast<uintptr_t>(x) & 15) != 0 || (reinterpret_cast<uintptr_t>(y) & 15) != 0 ||
        (reinterpret_cast<uintptr_t>(w) & 15) != 0)
        return -1;
    if (add && ((OH | OW) & 1 || (reinterpret_cast<uintptr_t>(add) & 15) != 0)) return -1;
    if (pool && (add || flip || OH != H || OW != W || ((H | W | PH | PW) & 1) || (reinterpret_cast<uintptr_t>(pool) & 15) != 0))
        return -1;
    const bool wide_tile = tz_wide_tile(B, OW);
    // 16 channels per workgroup (two per wavefront) while the operand registers allow it, else 8
    constexpr int CS = (2 * 4 * TzShape<K, 16, 16>::NM + 2 * 4 * TzShape<K, 16, 16>::RING) <= 160 ? 16 : 8;
    if (wide_tile) return launch_tz<T, K, 16, CS>(x, w, add, pool, y, B, H, W, C, PH, PW, flip, gate, s);
    return launch_tz<T, K, 8, CS>(x, w, add, pool, y, B, H, W, C, PH, PW, flip, gate, s);
}

template <int K>
static int launch_tz_dtype(const void* x, const void* w, const void* add, void* pool, void* y, int B, int H, int W, int C,
                           int PH, int PW, bool flip, int dtype, const TzGate* gate, hipStream_t s) {
    switch (dtype) {
        case kF16: return launch_tz_best<f16_t, K>(x, w, add, pool, y, B, H, W, C, PH, PW, flip, gate, s);
        case kBF16: return launch_tz_best<bf16_t, K>(x, w, add, pool, y, B, H, W, C, PH, PW, flip, gate, s);
        default: return -1;
    }
}

}  // namespace pdw
