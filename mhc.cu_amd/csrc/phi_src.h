// The caller's fp32 parameters, read by the kernel that multiplies with them (proj_fwd.hip, layer_fwd_onepass.hip).
#pragma once
#include "launchers.h"
#include "mhc_common.h"

namespace mhc {

// The caller's fp32 parameters, read by the projection itself (PF32 of the kernels): projection row d is a row of one of the three
// matrices, rounded to bf16 on its way into the LDS tile; some of the workgroups also store the rounded rows, [bias] and
// [alpha] for the kernels that follow and for the backward call.  Saves a packing launch (about 3 us of device and 5 us of host time per call, and for n = 32
// a read of the 89 MB that it wrote).
struct PhiSrc {
    const float *phi[3];
    const float *b[3], *alpha[3];
    void *phi_out;  // in the compute type: bf16, or fp32 in the exact tier
    float *bias_out, *alpha_out;
    int n;
};
__device__ __forceinline__ const float *phi_src_row(const PhiSrc &g, int d, int nC) {
    const float *base = d < g.n ? g.phi[0] : (d < 2 * g.n ? g.phi[1] : g.phi[2]);
    const int r = d < g.n ? d : (d < 2 * g.n ? d - g.n : d - 2 * g.n);
    return base + (size_t)r * nC;
}
__device__ __forceinline__ void gather_small(const PhiSrc &g, int tid, int nthr, int D) {
    if (tid < 3) g.alpha_out[tid] = g.alpha[tid][0];
    for (int i = tid; i < D; i += nthr)
        g.bias_out[i] = i < g.n ? g.b[0][i] : (i < 2 * g.n ? g.b[1][i - g.n] : g.b[2][i - 2 * g.n]);
}
inline PhiSrc phi_src_of(const ParamGather &g, int n) {
    PhiSrc s;
    for (int i = 0; i < 3; i++) {
        s.phi[i] = static_cast<const float *>(g.phi[i]);
        s.b[i] = g.b[i];
        s.alpha[i] = g.alpha[i];
    }
    s.phi_out = g.phi_out; s.bias_out = g.bias_out; s.alpha_out = g.alpha_out;
    s.n = n;
    return s;
}

}  // namespace mhc
