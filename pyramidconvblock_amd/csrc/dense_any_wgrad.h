// The weight gradient of dense_any.hip as a device function, so that dense_wide.hip can run it beside the row product that reads
// the same gradient; the matrix instructions and buffer loads it shares with the row kernel there.
#pragma once
#include "common.h"

namespace pdw {

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

// Per element type: the k values one step covers (a lane holds half of them, 16 bytes, consecutive) and the product.
template <typename T>
struct AnyStep;
template <>
struct AnyStep<float> {
    static constexpr int KS = 8;
    static __device__ __forceinline__ v16f mul(const uint4& a, const uint4& b, v16f c) {
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(__builtin_bit_cast(float, a.x), __builtin_bit_cast(float, b.x), c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(__builtin_bit_cast(float, a.y), __builtin_bit_cast(float, b.y), c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(__builtin_bit_cast(float, a.z), __builtin_bit_cast(float, b.z), c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(__builtin_bit_cast(float, a.w), __builtin_bit_cast(float, b.w), c, 0, 0, 0);
        return c;
    }
};
template <>
struct AnyStep<bf16_t> {
    static constexpr int KS = 16;
    static __device__ __forceinline__ v16f mul(const uint4& a, const uint4& b, v16f c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
    }
};
template <>
struct AnyStep<f16_t> {
    static constexpr int KS = 16;
    static __device__ __forceinline__ v16f mul(const uint4& a, const uint4& b, v16f c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
    }
};

typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));

// Loads go through buffer descriptors: an offset past the descriptor's end reads as zero and moves no data, so rows
// past the tensor and values past a row's end need no branch (a vector-memory instruction behind a branch makes the
// compiler wait for every load in flight).  kPast added to any offset of a descriptor of less than 2^31 bytes stays
// past its end.
constexpr uint32_t kPast = 0x80000000u;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t any_rsrc(const void* p, long long bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}

// Partials of dW[M][NO] = A^T B over row chunks: a workgroup makes a group of 4 tiles (a wavefront: one 32 x 32
// tile of dW for the chunk's rows).  The MFMA k is the row index: a lane holds one feature of 4 (fp32) or 8 (16-bit)
// rows, so consecutive lanes read consecutive features of a row.
struct AnyWgradArgs {
    const void *a, *b;
    float* part;
    int N, M, NO, rows_per_chunk, nt;   // nt: tiles along NO
    int chunks;
};

template <typename T>
__device__ __forceinline__ void dense_any_wgrad_body(const AnyWgradArgs& g, int chunk, int group) {
    const T* const A = (const T*)g.a;
    const T* const Bm = (const T*)g.b;
    float* const part = g.part;
    const int N = g.N, M = g.M, NO = g.NO, rows_per_chunk = g.rows_per_chunk, nt = g.nt;
    constexpr int KS = AnyStep<T>::KS, KL = KS / 2, ES = (int)sizeof(T);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l32 = lane & 31, h = lane >> 5;
    const int mt_total = (M + 31) / 32;
    const int tile = group * 4 + wave;
    if (tile >= mt_total * nt) return;
    const int tm = tile / nt, tn = tile - tm * nt;
    const long long rb = (long long)chunk * rows_per_chunk;
    const int nrows = (int)(rb + rows_per_chunk < N ? rows_per_chunk : N - rb);
    const int m = tm * 32 + l32, n = tn * 32 + l32;
    // descriptors over the chunk's rows: rows past the chunk read as zero; so does a feature past the width
    const __amdgpu_buffer_rsrc_t arsrc = any_rsrc(A + rb * M, (long long)nrows * M * ES);
    const __amdgpu_buffer_rsrc_t brsrc = any_rsrc(Bm + rb * NO, (long long)nrows * NO * ES);
    const uint32_t aoff = m < M ? (uint32_t)((KL * h * M + m) * ES) : kPast;
    const uint32_t boff = n < NO ? (uint32_t)((KL * h * NO + n) * ES) : kPast;
    v16f acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
    // one step: rows r .. r + KS - 1 of the chunk, this lane's are r + KL h .. + KL - 1
    auto fetch = [&](int r, uint4& a, uint4& b) {
        if constexpr (ES == 4) {
            uint32_t av[4], bv[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                av[t] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_raw_buffer_load_b32(arsrc, (int)(aoff + (uint32_t)((r + t) * M * ES)), 0, 0));
                bv[t] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_raw_buffer_load_b32(brsrc, (int)(boff + (uint32_t)((r + t) * NO * ES)), 0, 0));
            }
            a = make_uint4(av[0], av[1], av[2], av[3]);
            b = make_uint4(bv[0], bv[1], bv[2], bv[3]);
        } else {
            uint32_t av[8], bv[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                av[t] = (uint32_t)(unsigned short)__builtin_amdgcn_raw_buffer_load_b16(arsrc, (int)(aoff + (uint32_t)((r + t) * M * ES)), 0, 0);
                bv[t] = (uint32_t)(unsigned short)__builtin_amdgcn_raw_buffer_load_b16(brsrc, (int)(boff + (uint32_t)((r + t) * NO * ES)), 0, 0);
            }
            a = make_uint4(av[0] | (av[1] << 16), av[2] | (av[3] << 16), av[4] | (av[5] << 16), av[6] | (av[7] << 16));
            b = make_uint4(bv[0] | (bv[1] << 16), bv[2] | (bv[3] << 16), bv[4] | (bv[5] << 16), bv[6] | (bv[7] << 16));
        }
    };
    constexpr int D = 4;
    uint4 a[D], b[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
        fetch(d * KS, a[d], b[d]);
        __builtin_amdgcn_sched_barrier(0);   // (requested in the order in which the loop re-requests them)
    }
    for (int r = 0; r < nrows; r += D * KS) {   // (steps past the chunk multiply zeros)
#pragma unroll
        for (int d = 0; d < D; ++d) {
            acc = AnyStep<T>::mul(a[d], b[d], acc);
            fetch(r + (d + D) * KS, a[d], b[d]);
            // (keeps the steps in order: moved together, the loads of all steps end up behind all products, and the
            // next round then waits for every one of them instead of the oldest)
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // lane: column n of dW, rows tm * 32 + 8 (i / 4) + 4 h + i % 4
    float* po = part + (long long)chunk * M * NO;
    if (n < NO) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int mm = tm * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
            if (mm < M) po[(long long)mm * NO + n] = acc[i];
        }
    }
}

}  // namespace

// Row chunks of the weight gradient: enough wavefronts for the chip, at most `max_chunks` partials.
inline int any_wgrad_chunks(long long N, int M, int NO, int max_chunks) {
    const int tiles = ((M + 31) / 32) * ((NO + 31) / 32);
    long long c = (2048 + tiles - 1) / tiles;
    const long long by_rows = (N + 63) / 64;   // 64 rows per chunk at least
    if (c > by_rows) c = by_rows;
    if (c > max_chunks) c = max_chunks;
    return (int)(c < 1 ? 1 : c);
}

// The arguments of a weight gradient (N > 0) of at most max_chunks partials; false: offsets into a chunk beyond 32 bits.
inline bool any_wgrad_args(AnyWgradArgs& g, const void* a, const void* b, void* ws, long long N, int M, int NO, int dtype, int max_chunks) {
    const int chunks0 = any_wgrad_chunks(N, M, NO, max_chunks), ks = dtype == kF32 ? 8 : 16;
    long long rpc = (N + chunks0 - 1) / chunks0;
    rpc = (rpc + ks - 1) / ks * ks;
    g = AnyWgradArgs{a, b, (float*)ws, (int)N, M, NO, (int)rpc, (NO + 31) / 32, (int)((N + rpc - 1) / rpc)};
    return rpc * (M > NO ? M : NO) * (dtype == kF32 ? 4 : 2) <= 0x7fffffffLL;
}
inline int any_wgrad_groups(const AnyWgradArgs& g) { return ((g.M + 31) / 32 * g.nt + 3) / 4; }

}  // namespace pdw
