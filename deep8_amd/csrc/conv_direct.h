// Conv2d on an image of few channels without a patch matrix (conv_direct.hip).
#ifndef DEEP8_AMD_CONV_DIRECT_H
#define DEEP8_AMD_CONV_DIRECT_H

#include "common.h"

namespace d8 {

struct DirectShape {
    int B, IH, IW, C, OC, FH, FW, OH, OW, sy, sx, dy, dx, pt, pl;
};

// Whether the kernels take this layer: Float32 / Float16, dilation 1 along x, and a patch row that, with each of its FH
// runs of FW * C elements filled up to 16-byte pieces, fits the registers a wave keeps the filter in.
bool conv_direct_eligible(int dtype, const DirectShape &s);
// Microseconds that an eligible layer is expected to take on them (the gradient: infinite where ws_bytes do not hold the partial
// sums of one workgroup per 64 output channels).
double conv_direct_forward_us(int dtype, const DirectShape &s, const void *x);
double conv_direct_grad_us(int dtype, const DirectShape &s, const void *x, const void *gz, size_t ws_bytes);
// Partial sums of all the workgroups that the gradient would have.
size_t conv_direct_grad_bytes(int dtype, const DirectShape &s);
// z = conv(x, w) [+ bias] [relu]; round_first as GemmArgs::round_first.
int conv_direct_forward(int dtype, const DirectShape &s, const void *x, const void *w, void *z, const void *bias, int relu,
                        int round_first, hipStream_t stream);
// gw = beta * gw + the filter gradient.  ws takes the partial sums (fp32); false, with nothing launched, where not even
// those of one workgroup per 64 output channels fit.
bool conv_direct_grad_y(int dtype, const DirectShape &s, const void *x, void *gw, const void *gz, float beta, void *ws,
                        size_t ws_bytes, hipStream_t stream, int *rc);

}  // namespace d8

#endif
