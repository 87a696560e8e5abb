// Depthwise-convolution weight gradient on the dense matrix cores, 16-bit types, phase-major (dwconv_wgrad_ph.h).  Instantiations,
// workspace query and launchers, for one problem and for two of the same filter size in one launch.
#include "dwconv_wgrad_ph.h"

#include "reduce_parts.h"

namespace pdw {

size_t dwconv_wgrad_tz_workspace(int B, int H, int W, int C, int K, int PH, int PW, int dtype) {
    if (dtype == kF32) return 0;
    const WgPhPlan p = wgrad_ph_plan(B, H, W, C, K, PH, PW);
    return p.ok ? (size_t)p.parts() * K * K * C * sizeof(float) : 0;
}

static bool aligned(std::initializer_list<const void*> ptrs) {
    for (const void* p : ptrs)
        if (reinterpret_cast<uintptr_t>(p) & 15) return false;
    return true;
}

static int reduce(const void* ws, void* dw, int nparts, int n, int dtype, hipStream_t s) {
    return dtype == kF16 ? wgrad_reduce_launch<f16_t>((const float*)ws, dw, nparts, n, s)
                         : wgrad_reduce_launch<bf16_t>((const float*)ws, dw, nparts, n, s);
}

template <typename T>
static int wgrad_ph_go(const WgPhPlan& p, const void* x, const void* gy, void* ws, hipStream_t s) {
    if (wgrad_ph_ncopy(p.g.K) == 2) return launch_wgrad_ph<T, 2, 4>(p, x, gy, ws, s);
    return wgrad_ph_gr(p.g.K) == 4   ? launch_wgrad_ph<T, 3, 4>(p, x, gy, ws, s)
           : wgrad_ph_gr(p.g.K) == 2 ? launch_wgrad_ph<T, 3, 2>(p, x, gy, ws, s)
                                     : launch_wgrad_ph<T, 3, 8>(p, x, gy, ws, s);
}

template <typename T>
static int wgrad_ph_pair_go(const WgPhPlan& p0, const void* x0, const void* gy0, void* ws0, const WgPhPlan& p1, const void* x1,
                            const void* gy1, void* ws1, hipStream_t s) {
    const int K = p0.g.K;
    if (wgrad_ph_ncopy(K) == 2) return launch_wgrad_ph_pair<T, 2, 4>(p0, x0, gy0, ws0, p1, x1, gy1, ws1, s);
    return wgrad_ph_gr(K) == 4   ? launch_wgrad_ph_pair<T, 3, 4>(p0, x0, gy0, ws0, p1, x1, gy1, ws1, s)
           : wgrad_ph_gr(K) == 2 ? launch_wgrad_ph_pair<T, 3, 2>(p0, x0, gy0, ws0, p1, x1, gy1, ws1, s)
                                 : launch_wgrad_ph_pair<T, 3, 8>(p0, x0, gy0, ws0, p1, x1, gy1, ws1, s);
}

// -1: not covered (the caller falls back to the other weight-gradient kernels).
int dwconv_wgrad_tz_launch(const void* x, const void* gy, void* dw, void* ws, int B, int H, int W, int C, int K, int PH,
                           int PW, int dtype, hipStream_t s) {
    if (dtype == kF32 || !aligned({x, gy, ws})) return -1;
    const WgPhPlan p = wgrad_ph_plan(B, H, W, C, K, PH, PW);
    if (!p.ok) return -1;
    const int r = dtype == kF16 ? wgrad_ph_go<f16_t>(p, x, gy, ws, s) : wgrad_ph_go<bf16_t>(p, x, gy, ws, s);
    return r != 0 ? r : reduce(ws, dw, p.parts(), K * K * C, dtype, s);
}

// -1: not covered (the caller runs the two problems one by one).  Problem 0 is the wider one.
int dwconv_wgrad_tz_pair_launch(const void* x0, const void* gy0, void* dw0, void* ws0, int H0, int W0, const void* x1,
                                const void* gy1, void* dw1, void* ws1, int H1, int W1, int B, int C, int K, int PH, int PW,
                                int dtype, hipStream_t s) {
    if (dtype == kF32 || !aligned({x0, gy0, ws0, x1, gy1, ws1})) return -1;
    const WgPhPlan p0 = wgrad_ph_plan(B, H0, W0, C, K, PH, PW), p1 = wgrad_ph_plan(B, H1, W1, C, K, PH, PW);
    if (!p0.ok || !p1.ok) return -1;
    const int r = dtype == kF16 ? wgrad_ph_pair_go<f16_t>(p0, x0, gy0, ws0, p1, x1, gy1, ws1, s)
                                : wgrad_ph_pair_go<bf16_t>(p0, x0, gy0, ws0, p1, x1, gy1, ws1, s);
    const int n0 = p0.parts(), n1 = p1.parts();
    if (r != 0) return r;
    if (int e = reduce(ws0, dw0, n0, K * K * C, dtype, s)) return e;
    return reduce(ws1, dw1, n1, K * K * C, dtype, s);
}

}  // namespace pdw
