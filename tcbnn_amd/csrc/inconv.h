// What the first layer's kernels share: the problem and the matrix-core kernels' entry points.
#pragma once

#include "common.h"

namespace tcbnn {

struct InConvParams {
    const float* in;       // [B][3][H][W]
    const uint4* masks;    // [taps][opad32] {m0, m1, m2, pattern}, then the patterns alone: uint32 [taps][opad32]
    const float* bn;
    uint32_t* out;         // [OH][OW][ow][B]
    int32_t* res;          // residual tensor in format res_fmt, or null
    int res_fmt;           // TCBNN_RES_*
    int H, W, B, O, opad, ow;
    int R, S, stride_h, stride_w, pad_h, pad_w;
    int PH, PW, pool_h, pool_w, OH, OW;
};

// First layer on the matrix cores (inconv_mfma.hip): its kernel's name (false: it does not serve the problem), its launch
// (`served`: whether it does; if not, nothing has been launched).
bool inconv_mfma_kernel_name(const InConvParams& p, char* buf, size_t len);
int launch_inconv_mfma(const InConvParams& p, hipStream_t stream, bool* served);
// The kernel that it leaves few rows of 11x11 filters to (inconv_mfma_ring.hip); `dev` below kInConvDevices
constexpr int kInConvDevices = 64;
bool inconv_mfma_ring_serves(const InConvParams& p);
int launch_inconv_mfma_ring(const InConvParams& p, int dev, int cus, hipStream_t stream, bool* served);

}  // namespace tcbnn
