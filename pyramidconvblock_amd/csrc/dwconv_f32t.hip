// Dispatch of the fp32 depthwise convolutions on the fp32 matrix cores (dwconv_f32t.h, dwconv_wgrad_f32t.h) by filter size.
#include "dwconv_wgrad_f32t.h"

namespace pdw {

#define PDW_DECL(K)                                                                                                        \
    int dwconv_f32t_k##K(const void* x, const void* w, const void* add, void* y, int B, int H, int W, int C, int PH,       \
                         int PW, bool flip, int AH, int AW, hipStream_t s);                                                \
    int dwconv_f32t_pair_k##K(const void* x0, const void* w0, void* y0, int H0, int W0, const void* x1, const void* w1,    \
                              void* y1, int H1, int W1, int B, int C, hipStream_t s);                                      \
    int dwconv_wgrad_f32t_k##K(const void* x, const void* gy, void* dw, void* ws, int B, int H, int W, int C, int PH,      \
                               int PW, hipStream_t s);                                                                     \
    int dwconv_wgrad_f32t_pair_k##K(const void* x0, const void* gy0, void* dw0, void* ws0, int H0, int W0, const void* x1, \
                                    const void* gy1, void* dw1, void* ws1, int H1, int W1, int B, int C, int P, hipStream_t s,        \
                                    const MeanJob* mean, const void* w1, void* dx1);
PDW_DECL(3) PDW_DECL(5) PDW_DECL(7) PDW_DECL(9) PDW_DECL(11) PDW_DECL(13) PDW_DECL(15) PDW_DECL(17)
#undef PDW_DECL

#define PDW_BY_SIZE(CALL) \
    switch (K) {          \
        case 3: return CALL(3); \
        case 5: return CALL(5); \
        case 7: return CALL(7); \
        case 9: return CALL(9); \
        case 11: return CALL(11); \
        case 13: return CALL(13); \
        case 15: return CALL(15); \
        case 17: return CALL(17); \
        default: return -1; \
    }

int dwconv_f32t_launch(const void* x, const void* w, const void* add, void* y, int B, int H, int W, int C, int K, int PH, int PW,
                       bool flip, int AH, int AW, hipStream_t s) {
#define CALL(N) dwconv_f32t_k##N(x, w, add, y, B, H, W, C, PH, PW, flip, AH, AW, s)
    PDW_BY_SIZE(CALL)
#undef CALL
}

int dwconv_f32t_pair_launch(const void* x0, const void* w0, void* y0, int H0, int W0, const void* x1, const void* w1, void* y1, int H1,
                            int W1, int B, int C, int K, hipStream_t s) {
#define CALL(N) dwconv_f32t_pair_k##N(x0, w0, y0, H0, W0, x1, w1, y1, H1, W1, B, C, s)
    PDW_BY_SIZE(CALL)
#undef CALL
}

size_t dwconv_wgrad_f32t_workspace(int B, int H, int W, int C, int K, int PH, int PW) {
    const WgF32Plan p = wgrad_f32t_plan(B, H, W, C, K, PH, PW);
    return p.ok ? (size_t)p.nchunks * K * K * C * sizeof(float) : 0;
}

int dwconv_wgrad_f32t_launch(const void* x, const void* gy, void* dw, void* ws, int B, int H, int W, int C, int K, int PH, int PW,
                             hipStream_t s) {
#define CALL(N) dwconv_wgrad_f32t_k##N(x, gy, dw, ws, B, H, W, C, PH, PW, s)
    PDW_BY_SIZE(CALL)
#undef CALL
}

int dwconv_wgrad_f32t_pair_launch(const void* x0, const void* gy0, void* dw0, void* ws0, int H0, int W0, const void* x1,
                                  const void* gy1, void* dw1, void* ws1, int H1, int W1, int B, int C, int K, int P, hipStream_t s,
                                  const MeanJob* mean, const void* w1, void* dx1) {
#define CALL(N) dwconv_wgrad_f32t_pair_k##N(x0, gy0, dw0, ws0, H0, W0, x1, gy1, dw1, ws1, H1, W1, B, C, P, s, mean, w1, dx1)
    PDW_BY_SIZE(CALL)
#undef CALL
}

}  // namespace pdw
