// Dispatch of the block's three independent backward convolution launches as one (dwconv_bwd3.h) by filter size.
#include "common.h"
#include "kernels.h"
#include "mean_any.h"

namespace pdw {

// What the public call takes: the full scale in the wide tiles of both kernels, whole 16-channel slices.
bool dwconv_bwd3_covers(int B, int W, int C) {
    return C % 16 == 0 && W > 32 && (long long)cdiv(W, 64) * 64 * B <= (long long)cdiv(W, 32) * 32 * cdiv(B, 2) * 2;
}

#define PDW_BWD3_DECL(K)                                                                                               \
    int dwconv_bwd3_k##K(const void* gyf, const void* w0, const void* addp, void* dx, const void* x0, void* dw0, void* ws0, \
                         const void* x1, const void* gy1, void* dw1, void* ws1, int B, int H, int W, int h, int w, int C, \
                         int dtype, hipStream_t s, int* plan_out, const MeanJob* mean);
PDW_BWD3_DECL(3) PDW_BWD3_DECL(5) PDW_BWD3_DECL(7) PDW_BWD3_DECL(9) PDW_BWD3_DECL(11) PDW_BWD3_DECL(13) PDW_BWD3_DECL(15)
PDW_BWD3_DECL(17)
#undef PDW_BWD3_DECL

// -1: not covered (the caller makes the three launches).  With plan_out the launch is only planned: the band counts
// of the input gradient, the full and the half scale's weight gradient go to plan_out[0..2], no pointer is followed
// and nothing is launched; -1 then also where a given addp is better added by a launch of its own.
int dwconv_bwd3_launch(const void* gyf, const void* w0, const void* addp, void* dx, const void* x0, void* dw0, void* ws0,
                       const void* x1, const void* gy1, void* dw1, void* ws1, int B, int H, int W, int h, int w, int C, int K,
                       int dtype, hipStream_t s, int* plan_out, const MeanJob* mean) {
    if (tune_env("PDW_NO_BWD3")) return -1;
    switch (K) {
#define PDW_BWD3_CASE(KK) \
    case KK: return dwconv_bwd3_k##KK(gyf, w0, addp, dx, x0, dw0, ws0, x1, gy1, dw1, ws1, B, H, W, h, w, C, dtype, s, plan_out, mean);
        PDW_BWD3_CASE(3) PDW_BWD3_CASE(5) PDW_BWD3_CASE(7) PDW_BWD3_CASE(9) PDW_BWD3_CASE(11) PDW_BWD3_CASE(13)
        PDW_BWD3_CASE(15) PDW_BWD3_CASE(17)
#undef PDW_BWD3_CASE
        default: return -1;
    }
}

}  // namespace pdw
