// The four weights of a block whose halves of inner channels are padded to a multiple of 8 (block_any.hip), in the padded
// layout, eight values to a thread: conv_up's rows, conv_out's columns, the filters' channels.  A few hundred KB, 2.6 MB at 1144 channels: a launch of its
// own was latency (us of inference as a graph, with it and in the launch of the pool, conv_up reading its weights as they are given:
// [4,33,33,104] filter 9 37.1 -> 32.7, [3,57,61,200] filter 9 40.7 -> 36.4, [32,14,14,968] filter 3 71.2 -> 66.6).
#pragma once
#include "common.h"

namespace pdw {

struct PackArgs {
    const uint16_t *up, *out, *dw0, *dw1;
    uint16_t *up_p, *out_p, *dw0_p, *dw1_p;
    int D, G, Gp;
    int n_up, n_out, n_dw;   // vectors of 8 in each region
};

inline int pack_workgroups(const PackArgs& g) { return cdiv(g.n_up + g.n_out + 2 * g.n_dw, 256); }

__device__ __forceinline__ void pack_weights_body(const PackArgs& g, int wg) {   // (256 threads)
    int v = wg * 256 + threadIdx.x;
    const int I = 2 * g.G, Ip = 2 * g.Gp;
    if (v < g.n_up) {
        const int per = g.D / 8, row = v / per, c = v - row * per;
        const int hi = row >= g.Gp, r = row - hi * g.Gp;
        uint4 x = make_uint4(0, 0, 0, 0);
        if (r < g.G) x = *reinterpret_cast<const uint4*>(g.up + (long long)(hi * g.G + r) * g.D + c * 8);
        *reinterpret_cast<uint4*>(g.up_p + (long long)v * 8) = x;
        return;
    }
    v -= g.n_up;
    const uint16_t* src = g.out;
    uint16_t* dst = g.out_p;
    if (v >= g.n_out) {
        v -= g.n_out;
        src = g.dw0, dst = g.dw0_p;
        if (v >= g.n_dw) {
            v -= g.n_dw;
            src = g.dw1, dst = g.dw1_p;
            if (v >= g.n_dw) return;
        }
    }
    const int per = Ip / 8, row = v / per, c = (v - row * per) * 8;
    const int hi = c >= g.Gp, r = c - hi * g.Gp;
    ChanVec<uint16_t, 8> o;
#pragma unroll
    for (int i = 0; i < 8; ++i) o.v[i] = r + i < g.G ? src[(long long)row * I + hi * g.G + r + i] : (uint16_t)0;
    *reinterpret_cast<ChanVec<uint16_t, 8>*>(dst + (long long)v * 8) = o;
}

}  // namespace pdw
