// unet_kernels.hpp -- launch interface between the U-Net's host runtime
// (unet.cpp) and its gfx950 kernels (unet_kernels.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

typedef uint16_t bf16_t;

namespace unetk {

// where the gradient of a convolution's input goes: to the tensor itself, through
// the upsampling to one of half the resolution (sum of four), or through the
// average pooling to one of twice the resolution (a quarter to each of four, added
// to the skip connection's gradient)
enum BwdKind { BWD_SAME = 0, BWD_UP = 1, BWD_POOL = 2 };

// sums of partials (grad_reduce_kernel): out[e] = sum over c < chunks of
// part[c*n + e], e < n; first: first workgroup of every sum (32 elements each)
struct SumList {
    const float *part[32];
    float *out[32];
    int n[32], chunks[32], first[33];
    int count;
};

// every layer's masters, gradients, moments and packed copies (adam_kernel)
struct AdamLayer {
    float *w, *g, *m, *v, *b, *gb, *mb, *vb;
    bf16_t *wt, *wd;
    int Cout, Cin, first;   // first workgroup
};
struct AdamList {
    AdamLayer l[16];
    int count;
};

}  // namespace unetk

extern "C" {
hipError_t cffc_unet_launch_mfma_layout(float *out, hipStream_t st);
// workgroup tiles of a convolution with Cout output channels: the rows of dbp
int cffc_unet_conv_tiles(int B, int H, int W, int Cout);
// partials that the weight gradient writes
int cffc_unet_wgrad_chunks(int B, int H, int W, int Cin, int Cout);
hipError_t cffc_unet_launch_conv_fwd(const bf16_t *xA, int CA, int upA, const bf16_t *xB, int CB, int B, int H, int W,
                                     const bf16_t *wt, const float *bias, int Cout, int relu, bf16_t *y, float *y4,
                                     bf16_t *pool, hipStream_t st);
hipError_t cffc_unet_launch_conv_bwd_data(const bf16_t *G, int C, int B, int H, int W, const bf16_t *wd, int Cout,
                                          int CT, int kind, const bf16_t *act, bf16_t *Gt, float *dbp, float *gB,
                                          const float *gskip, hipStream_t st);
hipError_t cffc_unet_launch_conv_bwd_weight(const bf16_t *G, int Cout, const bf16_t *xA, int CA, int upA,
                                            const bf16_t *xB, int CB, int B, int H, int W, float *part,
                                            hipStream_t st);
hipError_t cffc_unet_launch_reduce(const unetk::SumList *L, hipStream_t st);
hipError_t cffc_unet_launch_mse(const float *y4, const float *t, int64_t P, int nwg, bf16_t *G, float *dbp,
                                float *lossp, hipStream_t st);
hipError_t cffc_unet_launch_adam(const unetk::AdamList *A, int nwg, float lr, float b1, float b2, float eps,
                                 float c1, float c2, int update, hipStream_t st);
hipError_t cffc_unet_launch_gather(const void *src, const int32_t *idx, int nrows, int64_t row_bytes, void *dst,
                                   hipStream_t st);
hipError_t cffc_unet_launch_to_bf16(const float *src, bf16_t *dst, int64_t n, hipStream_t st);
}
