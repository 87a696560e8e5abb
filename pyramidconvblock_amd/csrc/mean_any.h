// The global-mean branch of a block (conv_block.py:46-49) for any width, as workgroup bodies of 256 threads that ride in
// the grids of the resampling launches around them: column sums of a tensor over ranges of an image's positions, and
// the two small products (mean -> conv_pool -> a row per image; its transpose).  16-byte vectors: widths that are
// multiples of 16 bytes.  Bandwidth for the sums, latency for the products: a product's workgroup takes 64 features of
// one image and adds up the image's partial sums itself, so that nothing has to wait for a summation launch; the plan
// keeps the partials few (32 an image at most) because every such workgroup reads them all.  At [4,64,64,1152] the four
// launches that this replaces (two sums, two products with up to 128 partials an image) took 10 + 24 + 10 + 52 us.
#pragma once
#include "common.h"
#include "pack_weights.h"

namespace pdw {

struct ColsumJob {
    const void* x;   // [B][P][C]
    float* part;     // [B][n][C]
    int B, P, C, n, len;      // n ranges of len positions
    int lanes_log, slices;    // 1 << lanes_log vectors of a row to a workgroup, slices of them
    bool pairs;               // colsum_body<T, true>: eight positions in pairs
};

inline int colsum_workgroups(const ColsumJob& j) { return j.B * j.n * j.slices; }

// part = nullptr: only the plan (for the size of the partials, which fewer workgroups never make larger).
inline ColsumJob colsum_plan(const void* x, float* part, int B, int P, int C, int esize, int workgroups = 512) {
    const int V = 16 / esize, vecs = C / V;
    ColsumJob j{x, part, B, P, C, 1, P, 3, 1, false};
    while (j.lanes_log < 5 && (1 << j.lanes_log) < vecs) ++j.lanes_log;
    j.slices = cdiv(vecs, 1 << j.lanes_log);
    const int pl = 256 >> j.lanes_log;
    int n = cdiv(workgroups, (long long)B * j.slices);   // two workgroups per compute unit ...
    if (n > P / (pl * 8)) n = P / (pl * 8);       // ... of at least eight positions a thread
    if (n > 32) n = 32;
    if (n < 1) n = 1;
    j.len = cdiv(P, n), j.n = cdiv(P, j.len);
    return j;
}

// red: 256 * V floats of LDS (V = values per 16 bytes).  PAIRS, for jobs that say so: of every eight positions pairs, then pairs of those, before
// they are added to the sum (as many additions): where ranges are longer because fewer workgroups ride along, a thread's chain of roundings is
// shorter all the same (error of the sums over 100352 rows of 128 in fp32, 2-norm: 512 workgroups 1.35e-7, 192 1.8e-7, 192 in pairs 1.24e-7).
template <typename T, bool PAIRS = false>
__device__ __forceinline__ void colsum_body(const ColsumJob& j, int wg, float* red) {
    constexpr int V = 16 / (int)sizeof(T);
    const int sl = wg % j.slices, rest = wg / j.slices, ch = rest % j.n, b = rest / j.n;
    const int tid = threadIdx.x, lanes = 1 << j.lanes_log, cv = tid & (lanes - 1), pl = tid >> j.lanes_log, PL = 256 >> j.lanes_log;
    const int c = (sl * lanes + cv) * V;
    const int p1 = min((ch + 1) * j.len, j.P);
    float acc[V];
#pragma unroll
    for (int v = 0; v < V; ++v) acc[v] = 0.f;
    if (c < j.C) {
        const T* xb = (const T*)j.x + (long long)b * j.P * j.C + c;
        int p = ch * j.len + pl;
        for (; p + 7 * PL < p1; p += 8 * PL) {   // eight loads in flight
            ChanVec<T, V> xv[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) xv[u] = *reinterpret_cast<const ChanVec<T, V>*>(xb + (long long)(p + u * PL) * j.C);
            if (PAIRS && j.pairs) {   // (uniform)
#pragma unroll
                for (int v = 0; v < V; ++v) {
                    auto two = [&](int u) { return to_f32(xv[u].v[v]) + to_f32(xv[u + 1].v[v]); };
                    acc[v] += (two(0) + two(2)) + (two(4) + two(6));
                }
            } else {
#pragma unroll
                for (int u = 0; u < 8; ++u)
#pragma unroll
                    for (int v = 0; v < V; ++v) acc[v] += to_f32(xv[u].v[v]);
            }
        }
        for (; p < p1; p += PL) {
            float xv[V];
            load_f32<T, V>(xb + (long long)p * j.C, xv);
#pragma unroll
            for (int v = 0; v < V; ++v) acc[v] += xv[v];
        }
    }
#pragma unroll
    for (int v = 0; v < V; v += 4) *reinterpret_cast<float4*>(red + tid * V + v) = make_float4(acc[v], acc[v + 1], acc[v + 2], acc[v + 3]);
    __syncthreads();
    const int cols = lanes * V;   // <= 256
    if (tid < cols && sl * cols + tid < j.C) {
        float s = 0.f;
        for (int q = 0; q < PL; ++q) s += red[q * cols + tid];
        j.part[((long long)b * j.n + ch) * j.C + sl * cols + tid] = s;
    }
}

// sm[c] = sum over the n partials of an image, c < D; D % 4 == 0.  red: NT float4 of LDS.  Ends with a barrier.
template <int NT>
__device__ __forceinline__ void image_sums(const float* __restrict__ pp, int n, int D, float* sm, float4* red) {
    const int tid = threadIdx.x, d4 = D / 4;
    int L = 16;
    while (L < NT && L < d4) L <<= 1;
    const int cl = tid & (L - 1), ql = tid / L, QL = NT / L;
    for (int c0 = 0; c0 < d4; c0 += L) {   // (more than once only where QL = 1)
        const int c = c0 + cl;
        float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
        if (c < d4) {
            const float* p = pp + c * 4;
            int q = ql;
            for (; q + 7 * QL < n; q += 8 * QL) {
                float4 v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = *reinterpret_cast<const float4*>(p + (long long)(q + u * QL) * D);
#pragma unroll
                for (int u = 0; u < 8; ++u) s.x += v[u].x, s.y += v[u].y, s.z += v[u].z, s.w += v[u].w;
            }
            for (; q < n; q += QL) {
                const float4 v = *reinterpret_cast<const float4*>(p + (long long)q * D);
                s.x += v.x, s.y += v.y, s.z += v.z, s.w += v.w;
            }
        }
        if (QL == 1) {
            if (c < d4) *reinterpret_cast<float4*>(sm + c * 4) = s;
        } else {
            red[ql * L + cl] = s;
            __syncthreads();
            if (ql == 0 && c < d4) {
                for (int q = 1; q < QL; ++q) {
                    const float4 v = red[q * L + cl];
                    s.x += v.x, s.y += v.y, s.z += v.z, s.w += v.w;
                }
                *reinterpret_cast<float4*>(sm + c * 4) = s;
            }
        }
    }
    __syncthreads();
}

// The same for `images` <= IM images after one another (partials of few ranges: many images), into sm[image][D].
template <int NT, int IM>
__device__ __forceinline__ void images_sums(const float* __restrict__ pp, int n, int D, int images, float* sm) {
    const int d4 = D / 4;
    for (int i = threadIdx.x; i < IM * d4; i += NT) {
        const int im = i / d4, c = i - im * d4;
        float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
        if (im < images) {
            const float* p = pp + (long long)im * n * D + c * 4;
            int q = 0;
            for (; q + 3 < n; q += 4) {
                float4 v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) v[u] = *reinterpret_cast<const float4*>(p + (long long)(q + u) * D);
#pragma unroll
                for (int u = 0; u < 4; ++u) s.x += v[u].x, s.y += v[u].y, s.z += v[u].z, s.w += v[u].w;
            }
            for (; q < n; ++q) {
                const float4 v = *reinterpret_cast<const float4*>(p + (long long)q * D);
                s.x += v.x, s.y += v.y, s.z += v.z, s.w += v.w;
            }
        }
        *reinterpret_cast<float4*>(sm + i * 4) = s;
    }
    __syncthreads();
}

constexpr int kMeanOut = 64;   // features of a workgroup of the products
constexpr int kMeanImages = 4; // images of one in the backward, where there would be many

struct MeanJob {
    const float* part;   // [B][n][D]
    int n, B, D;
    float inv_p;
    const void *wp, *bp, *bo;
    void* m;             // forward: the mean
    float* rowbias;      // forward: m Wp^T + bp + bo
    float *gs, *dmean;   // backward: the sums of the gradient, their product with Wp over P
    bool shared;         // backward in dwconv_bwd3_k: kMeanImages images to a workgroup
};

inline int mean_slices(int D) { return cdiv(D, kMeanOut); }
// Whether a workgroup of the backward takes four images: where one each would make more workgroups than the convolutions' shared
// launch, which holds one workgroup a compute unit, has units left for.  They read the layer's weight once and take less than twice as long.  Training
// steps, us: [102,10,13,608] filter 9 bf16 (1020 workgroups -> 260) 249 -> 230, [40,7,7,1152] filter 5 184 -> 151, [20,14,14,1024] filter 5 (320
// -> 80) 147 -> 138, [64,20,20,256] (256 -> 64) 117 -> 113; with eight images [12,28,28,768] (144 -> 24) 156 -> 179.
inline bool mean_shared(int B, int D) { return (long long)B * mean_slices(D) > 192 && D > 128 && D <= 2048; }
inline int mean_bwd_workgroups(const MeanJob& j) { return cdiv(j.B, j.shared ? kMeanImages : 1) * mean_slices(j.D); }
// sums; scratch of 32 bytes a thread (backward, 16-bit) or less
inline size_t mean_lds(int D, int nt = 256, int images = 1) { return (size_t)images * D * sizeof(float) + (size_t)nt * 32; }

template <typename T>
__device__ __forceinline__ void mean_fwd_body(const MeanJob& j, int wg, float* sm) {
    constexpr int V = 16 / (int)sizeof(T);
    const int slices = (j.D + kMeanOut - 1) / kMeanOut, b = wg / slices, sl = wg - b * slices, D = j.D, tid = threadIdx.x;
    image_sums<256>(j.part + (long long)b * j.n * D, j.n, D, sm, reinterpret_cast<float4*>(sm + D));
    for (int c = tid; c < D; c += 256) {
        const T mv = from_f32<T>(sm[c] * j.inv_p);
        if (sl == 0) ((T*)j.m)[(long long)b * D + c] = mv;
        sm[c] = to_f32(mv);
    }
    __syncthreads();
    const int sub = tid & 7, nv = D / V;
#pragma unroll
    for (int pass = 0; pass < kMeanOut / 32; ++pass) {   // eight lanes to a feature
        const int o = sl * kMeanOut + pass * 32 + (tid >> 3);
        float acc = 0.f;
        if (o < D) {
            const T* wr = (const T*)j.wp + (long long)o * D;
            int v = sub;
            for (; v + 24 < nv; v += 32) {
                ChanVec<T, V> wv[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) wv[u] = *reinterpret_cast<const ChanVec<T, V>*>(wr + (v + 8 * u) * V);
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int e = 0; e < V; ++e) acc = fmaf(sm[(v + 8 * u) * V + e], to_f32(wv[u].v[e]), acc);
            }
            for (; v < nv; v += 8) {
                float wv[V];
                load_f32<T, V>(wr + v * V, wv);
#pragma unroll
                for (int e = 0; e < V; ++e) acc = fmaf(sm[v * V + e], wv[e], acc);
            }
        }
        acc += __shfl_xor(acc, 1);
        acc += __shfl_xor(acc, 2);
        acc += __shfl_xor(acc, 4);
        if (sub == 0 && o < D) {
            if (j.bp) acc += to_f32(((const T*)j.bp)[o]);
            if (j.bo) acc += to_f32(((const T*)j.bo)[o]);
            j.rowbias[(long long)b * D + o] = acc;
        }
    }
}

// The same by workgroups of half as many features each, with everything that can be in flight so: what takes the time is trips to memory one after the
// other.  Sixteen partials at once, the first weights requested before them, and eight at a time.  124 registers: for launches whose other
// workgroups are all on the chip with those too (gate_pair_mean_fwd_launch).
constexpr int kMeanFew = 32;
template <typename T>
__device__ __forceinline__ void mean_fwd_deep_body(const MeanJob& j, int wg, float* sm) {
    constexpr int V = 16 / (int)sizeof(T);
    typedef ChanVec<T, V> Vec;
    const int D = j.D, d4 = D / 4, slices = (D + kMeanFew - 1) / kMeanFew, b = wg / slices, sl = wg - b * slices, tid = threadIdx.x;
    const int sub = tid & 7, nv = D / V, o = sl * kMeanFew + (tid >> 3);
    // vector v of the thread's feature (past the end: the last one, which is not added)
    auto weight = [&](int v) { return *reinterpret_cast<const Vec*>((const T*)j.wp + (uint32_t)(min(o, D - 1) * D + min(v, nv - 1) * V)); };
    Vec pre[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) pre[u] = weight(sub + 8 * u);
    // sums: two columns of four a thread (c, c + L) over every QL-th partial; past the end the last one, not added
    {
        float4* const red = reinterpret_cast<float4*>(sm + D);
        const float* const pp = j.part + (long long)b * j.n * D;
        const int n = j.n, L = min((d4 + 1) / 2, 256), QL = 256 / L, ql = tid / L, cl = tid - ql * L;
        for (int c0 = 0; c0 < d4; c0 += 2 * L) {   // (more than once only where QL = 1)
            float4 s[2] = {make_float4(0.f, 0.f, 0.f, 0.f), make_float4(0.f, 0.f, 0.f, 0.f)};
            const int c1 = c0 + cl, c[2] = {min(c1, d4 - 1), min(c1 + L, d4 - 1)};
            if (ql < QL)
                for (int q = ql; q < n; q += 8 * QL) {
                    float4 v[8][2];
#pragma unroll
                    for (int u = 0; u < 8; ++u)
#pragma unroll
                        for (int k = 0; k < 2; ++k) v[u][k] = *reinterpret_cast<const float4*>(pp + (uint32_t)(min(q + u * QL, n - 1) * D + c[k] * 4));
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        if (q + u * QL < n) {
#pragma unroll
                            for (int k = 0; k < 2; ++k) s[k].x += v[u][k].x, s[k].y += v[u][k].y, s[k].z += v[u][k].z, s[k].w += v[u][k].w;
                        }
                }
            if (QL > 1) {
                if (ql < QL) red[ql * 2 * L + cl] = s[0], red[(ql * 2 + 1) * L + cl] = s[1];
                __syncthreads();
                if (ql == 0)
                    for (int q = 1; q < QL; ++q)
#pragma unroll
                        for (int k = 0; k < 2; ++k) {
                            const float4 v = red[(q * 2 + k) * L + cl];
                            s[k].x += v.x, s[k].y += v.y, s[k].z += v.z, s[k].w += v.w;
                        }
            }
            if (ql == 0) {
#pragma unroll
                for (int k = 0; k < 2; ++k)
                    if (c1 + k * L < min(d4, c0 + (k + 1) * L)) *reinterpret_cast<float4*>(sm + (c1 + k * L) * 4) = s[k];
            }
        }
        __syncthreads();
    }
    for (int c = tid; c < D; c += 256) {
        const T mv = from_f32<T>(sm[c] * j.inv_p);
        if (sl == 0) ((T*)j.m)[(long long)b * D + c] = mv;
        sm[c] = to_f32(mv);
    }
    __syncthreads();
    float acc = 0.f;   // (mean_fwd_body's order)
    auto add = [&](const Vec& w, int v) {
        if (v < nv) {
#pragma unroll
            for (int e = 0; e < V; ++e) acc = fmaf(sm[v * V + e], to_f32(w.v[e]), acc);
        }
    };
#pragma unroll
    for (int u = 0; u < 4; ++u) add(pre[u], sub + 8 * u);
    for (int v = sub + 32; v < nv; v += 64) {
        Vec wv[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) wv[u] = weight(v + 8 * u);
#pragma unroll
        for (int u = 0; u < 8; ++u) add(wv[u], v + 8 * u);
    }
    acc += __shfl_xor(acc, 1);
    acc += __shfl_xor(acc, 2);
    acc += __shfl_xor(acc, 4);
    if (sub == 0 && o < D) {
        if (j.bp) acc += to_f32(((const T*)j.bp)[o]);
        if (j.bo) acc += to_f32(((const T*)j.bo)[o]);
        j.rowbias[(long long)b * D + o] = acc;
    }
}

// By a workgroup of NT threads.
template <typename T, int NT, int IM>
__device__ __forceinline__ void mean_bwd_images(const MeanJob& j, int wg, float* sm) {
    constexpr int V = 16 / (int)sizeof(T), CL = kMeanOut / V, OL = NT / CL;   // column lanes, row lanes
    const int slices = (j.D + kMeanOut - 1) / kMeanOut, b0 = wg / slices * IM, sl = wg % slices, D = j.D, tid = threadIdx.x;
    const int images = min(IM, j.B - b0);
    float* red = sm + IM * D;   // [OL][64]
    const float* const part = j.part + (long long)b0 * j.n * D;
    if constexpr (IM == 1) image_sums<NT>(part, j.n, D, sm, reinterpret_cast<float4*>(red));
    else images_sums<NT, IM>(part, j.n, D, images, sm);
    if (sl == 0)
        for (int c = tid; c < images * D; c += NT) j.gs[(long long)b0 * D + c] = sm[c];
    const int cv = tid % CL, ol = tid / CL, c = sl * kMeanOut + cv * V;
    float acc[IM][V];
#pragma unroll
    for (int i = 0; i < IM; ++i)
#pragma unroll
        for (int e = 0; e < V; ++e) acc[i][e] = 0.f;
    if (c < D) {
        const T* wc = (const T*)j.wp + c;
        auto add = [&](const ChanVec<T, V>& wv, int o) {
#pragma unroll
            for (int i = 0; i < IM; ++i)
#pragma unroll
                for (int e = 0; e < V; ++e) acc[i][e] = fmaf(sm[i * D + o], to_f32(wv.v[e]), acc[i][e]);
        };
        int o = ol;
        for (; o + 7 * OL < D; o += 8 * OL) {
            ChanVec<T, V> wv[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) wv[u] = *reinterpret_cast<const ChanVec<T, V>*>(wc + (long long)(o + u * OL) * D);
#pragma unroll
            for (int u = 0; u < 8; ++u) add(wv[u], o + u * OL);
        }
        for (; o < D; o += OL) add(*reinterpret_cast<const ChanVec<T, V>*>(wc + (long long)o * D), o);
    }
#pragma unroll
    for (int i = 0; i < IM; ++i) {
        if (i > 0) __syncthreads();
#pragma unroll
        for (int e = 0; e < V; ++e) red[ol * kMeanOut + cv * V + e] = acc[i][e];
        __syncthreads();
        if (tid < kMeanOut && sl * kMeanOut + tid < D && i < images) {
            float t = 0.f;
            for (int q = 0; q < OL; ++q) t += red[q * kMeanOut + tid];
            j.dmean[(long long)(b0 + i) * D + sl * kMeanOut + tid] = t * j.inv_p;
        }
    }
}

// SHARED: where a job may have kMeanImages images to a workgroup (twice the instructions of one that never has).
template <typename T, int NT, bool SHARED>
__device__ __forceinline__ void mean_bwd_body(const MeanJob& j, int wg, float* sm) {
    if (SHARED && j.shared) mean_bwd_images<T, NT, kMeanImages>(j, wg, sm);   // (uniform)
    else mean_bwd_images<T, NT, 1>(j, wg, sm);
}

// Whether the bodies take the case (host side).
inline bool mean_any_ok(const void* x, const void* wp, const void* m, int D, int esize) {
    return D % (16 / esize) == 0 && D <= 8192 && (reinterpret_cast<uintptr_t>(x) & 15) == 0 && (reinterpret_cast<uintptr_t>(wp) & 15) == 0 &&
           (reinterpret_cast<uintptr_t>(m) & 15) == 0;
}

// dense_wide.hip: the block's first layer with the sums of its input and the 2 x 2 pool of its result
bool dense_wide_first_plan(ColsumJob* sums, long long N, int K, int NO, int B, int P, int dtype);
int dense_wide_first_launch(const void* x, const void* w, void* y, void* pool, int w_half, long long N, int K, int NO, const ColsumJob& sums,
                            const PackArgs* pack, int dtype, hipStream_t s);
// resample.hip: the launches that they ride in.
// xp = adaptive average pool of a to (h, w), with the column sums and the packing of weights that are given
int avgpool_with_launch(const void* a, void* xp, int B, int H, int W, int C, int h, int w, const ColsumJob* sums, const PackArgs* pack,
                        int dtype, hipStream_t s);
// gate_pair_fwd_launch with the mean branch's forward
int gate_pair_mean_fwd_launch(const void* xf, const void* xh, void* y, int B, int H, int W, int h, int w, int I, int ldy,
                              const MeanJob& mean, int dtype, hipStream_t s, int gw);
// gate_pair_bwd_launch with the column sums
int gate_pair_colsum_bwd_launch(const void* gy, const void* xf, const void* xh, void* gxf, void* gxh, int B, int H, int W, int h,
                                int w, int I, int ldg, const ColsumJob& sums, int dtype, hipStream_t s, int gw);
// the mean branch's backward: what its launch leaves to the deferred summations (the gradients of the pooled layer's weight
// and biases), and the launch of its own with that
int mean_bwd_defer(const MeanJob& mean, void* gbias, void* gbias2, void* gwp, int dtype, hipStream_t s);
int mean_bwd_launch(const MeanJob& mean, void* gbias, void* gbias2, void* gwp, int dtype, hipStream_t s);

}  // namespace pdw
