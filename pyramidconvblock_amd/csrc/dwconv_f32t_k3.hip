// fp32 depthwise convolution on the fp32 matrix cores, 3x3 filter: the instantiations of the kernel templates in
// dwconv_f32t.h (forward / input gradient) and dwconv_wgrad_f32t.h (weight gradient) for this size, one translation unit per
// size so the build compiles them in parallel.
#include "dwconv_f32t.h"
#include "dwconv_wgrad_f32t.h"

namespace pdw {

int dwconv_f32t_k3(const void* x, const void* w, const void* add, void* y, int B, int H, int W, int C, int PH, int PW, bool flip,
                   int AH, int AW, hipStream_t s) {
    return launch_f32t<3>(x, w, add, y, B, H, W, C, PH, PW, flip, AH, AW, s);
}

int dwconv_f32t_pair_k3(const void* x0, const void* w0, void* y0, int H0, int W0, const void* x1, const void* w1, void* y1, int H1,
                        int W1, int B, int C, hipStream_t s) {
    return launch_f32t_pair<3>(x0, w0, y0, H0, W0, x1, w1, y1, H1, W1, B, C, s);
}

int dwconv_wgrad_f32t_k3(const void* x, const void* gy, void* dw, void* ws, int B, int H, int W, int C, int PH, int PW,
                         hipStream_t s) {
    return launch_wgrad_f32t<3>(x, gy, dw, ws, B, H, W, C, PH, PW, s);
}

int dwconv_wgrad_f32t_pair_k3(const void* x0, const void* gy0, void* dw0, void* ws0, int H0, int W0, const void* x1,
                              const void* gy1, void* dw1, void* ws1, int H1, int W1, int B, int C, int P, hipStream_t s,
                              const MeanJob* mean, const void* w1, void* dx1) {
    return launch_wgrad_f32t_pair<3>(x0, gy0, dw0, ws0, H0, W0, x1, gy1, dw1, ws1, H1, W1, B, C, P, s, mean, w1, dx1);
}

}  // namespace pdw
