// nn.hpp -- launchers of the learned preconditioner's network kernels
// (nn_kernels.hip).  Grids are node counts per direction {x, y, z}.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace mfx {

// layer 0 (1 -> 16, FP32 input in32), 1..6 (BF16 MFMA), 7 (16 -> 1, FP32
// output out32); od: output grid, id: input tensor grid
void nn_conv_forward(int layer, const uint16_t *in, const float *in32, const uint16_t *wb,
                     const float *wr, const uint16_t *skip, uint16_t *out, float *out32,
                     const uint32_t *od, const uint32_t *id, hipStream_t s);
// Data gradient of layer 1..6 in slot order (nn_kernels.hip), masked by the
// input activation act > 0.  Layers 1-3 (stride 2; xd the input grid): out =
// add + the transposed convolution of G.  Layers 4-6 (od the fine grid of the
// up-sampled input, xd the coarse input grid): out = the transposed
// convolution summed over each coarse node's children; add unused.
// wa: the weights as nn_pack_weights orders them.
void nn_conv_adjoint(int layer, const float *G, const float *wa, const float *add,
                     const uint16_t *act, float *out, const uint32_t *od, const uint32_t *xd,
                     hipStream_t s);
// grad += dL/dW of all layers (G: output gradients in slot order, layer 7:
// dy; in: the layer's bf16 input, layer 0: nullptr with x32).  part: scratch
// of n_parts x n_weights floats per layer, n_parts = nn_wgrad_parts.
struct NnWgrad {
  const uint16_t *in;
  const float *G;
  float *part;
  const uint32_t *od, *id;
  uint32_t n_parts, n_weights;
};
uint32_t nn_wgrad_parts(int layer, const uint32_t *od);
void nn_wgrad(const NnWgrad (&l)[8], const float *x32, float *grad, hipStream_t s);
void nn_head_backward(const float *dy, const float *W, const uint16_t *act, float *g,
                      const uint32_t *d, hipStream_t s);
uint32_t nn_mse_blocks(uint64_t n);
void nn_mse(const float *y, const float *target, const uint8_t *mask, float scale, float *dy,
            double *part, uint64_t n, hipStream_t s);
void nn_adam(float *w, float *m, float *v, const float *g, uint32_t n, float lr, float b1, float b2,
             float eps, int step, hipStream_t s);
void nn_pack_weights(const float *w, uint16_t *wb, float *wr, float *wa, int cin, int cout, int kp,
                     hipStream_t s);
void nn_scale_to_f32(const double *r, float *out, double scale, uint64_t n, hipStream_t s);
void nn_scale_to_f64(const float *y, double *z, double scale, uint64_t n, hipStream_t s);
void nn_axpy_f32(float *x, float a, const float *y, uint64_t n, hipStream_t s);

}  // namespace mfx
