// nn_launch.hpp — host-side launchers of the warm-start network kernels
// (nn_kernels.hip).  BF16 tensors are passed as uint16_t storage.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lbmnn {

typedef uint16_t u16;

// Input of a 3x3 conv: NHWC tensor in0 (C0 channels, B x H x W), optionally
// concatenated with the nearest-upsampled NHWC tensor in1 (C1 channels,
// B x ceil(H/2) x ceil(W/2)).  C0 and C1 are multiples of 32.
struct ConvSrc {
  const u16* in0 = nullptr;
  int C0 = 0;
  const u16* in1 = nullptr;
  int C1 = 0;
  int B = 0, H = 0, W = 0;
  int dil = 1;  // dilation of the 3x3 stencil
};

// out = act(conv3x3(src, w) + bias), zero where mask (laid out as out) is not
// above zero; w is a [Cout][9][C0 + C1] that pack_w packed, bias and mask may
// be null.
hipError_t conv3x3(const ConvSrc& s, const u16* w, const float* bias, const u16* mask, u16* out,
                   int Cout, bool relu, hipStream_t st);
// Weight-gradient partial sums into part, [chunks][Cout][9][Cin]; with_bias:
// each chunk's block is followed by its Cout sums of the bias gradient
// (Cout, Cin multiples of 32).
struct WgradPlan {
  int chunks = 0;
  bool with_bias = false;
};
WgradPlan wgrad_plan(const ConvSrc& s, int Cout);
hipError_t wgrad(const ConvSrc& s, const u16* dout, int Cout, float* part, hipStream_t st);
hipError_t colsum_part(const u16* g, int P, int C, int px_per_chunk, float* part, hipStream_t st);
hipError_t reduce_chunks(const float* part, int nchunk, long n, float* out, hipStream_t st);
// wf: the BF16 weights of a conv, packed for conv3x3; wt: its data gradient's.
hipError_t pack_w(const float* w, u16* wf, u16* wt, int Cout, int Cin, hipStream_t st);
// Divergence penalty of the predicted velocity: d (per pixel) and its
// per-256-pixel sums of d^2 into part; dy += the gradient of (g / 2) sum d^2.
hipError_t div_penalty(const float* y, const float* mask, float* d, float* part, float* dy, int B,
                       int H, int W, float su, float sv, float g, hipStream_t st);
hipError_t pool(const u16* in, u16* out, int B, int H, int W, int C, hipStream_t st);
hipError_t skip_grad(const u16* dcat, int Ccat, const u16* dpool, const u16* s, u16* ds, int B,
                     int H, int W, int C, hipStream_t st);
hipError_t up_grad(const u16* dcat, int Ccat, int C0, const u16* y, u16* dy, int B, int H, int W,
                   int C1, hipStream_t st);
hipError_t head_fwd(const u16* x, const float* w, const float* b, float* out, int P, int C, int K,
                    hipStream_t st);
hipError_t mse(const float* y, const float* t, const float* mask, float* dy, float* part, int P,
               int K, float inv_norm, hipStream_t st);
hipError_t head_bwd(const float* dy, const float* w, const u16* x, u16* dx, int P, int C, int K,
                    hipStream_t st);
hipError_t head_wgrad_part(const float* dy, const u16* x, float* part, int P, int C, int K,
                           int px_per_chunk, hipStream_t st);
hipError_t adam(float* p, const float* g, float* m, float* v, long n, float lr, float b1, float b2,
                float eps, float c1, float c2, float wd, hipStream_t st);
hipError_t gather(const float* inputs, const float* targets, const int* idx, u16* x, float* t,
                  float* mask, int B, int HW, int Ci, int Cp, hipStream_t st);

}  // namespace lbmnn
