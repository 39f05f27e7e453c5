// pdt_cnn.hpp -- host entry points into the warm-start network kernels
// (pdt_cnn.hip).  Activations are NHWC; bf16 buffers are passed as void*.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace pdt {

// Layer shapes with kernels: 2 -> 32, 32 -> 32, 32 -> 6.
bool cnn_layer_supported(int cin, int cout);
// A layer as the kernels that take the whole network in one launch see it.
struct CnnLayer {
  const float* w;  // fp32 master W[tap][co][ci], b
  float* g;        // its gradient, same layout
  void* wk;        // packed bf16 weights
  void* wt;        // packed bf16 weights of the backward-data pass (null: first layer)
  float* part;     // per-block partial gradients (cnn_wgrad_part_floats)
  int cin, cout;
  int nblk;        // partials written by cnn_conv_wgrad
  int nk, nt;      // elements of wk, wt (set by cnn_pack_weights)
};
constexpr int kCnnLayers = 8;  // layers per launch
struct CnnLayers {
  CnnLayer l[kCnnLayers];
};

// Elements of the packed bf16 weights of a convolution cin -> cout (the
// backward-data pass of a layer is one of its output to its input channels).
size_t cnn_wk_elems(int cin, int cout);
// fp32 master weights -> packed bf16 copies.
void cnn_pack_weights(hipStream_t st, const CnnLayer* ls, int count);
// The layers of the forward pass: relu(conv(x) + b) in bf16 from the fp32
// input (2 -> 32), between hidden activations (32 -> 32), and the fp32
// output conv(in) + b (32 -> 6).
void cnn_conv_first(hipStream_t st, const float* x, const void* wk, const float* b, void* out, int n, int h, int w);
void cnn_conv_hidden(hipStream_t st, const void* in, const void* wk, const float* b, void* out, int n, int h, int w);
void cnn_conv_last(hipStream_t st, const void* in, const void* wk, const float* b, float* y, int n, int h, int w);
// The whole network in one launch, workgroups of `rows` output rows by a strip
// of columns; x and y must not overlap.  cnn_net_rows: the rows that make it
// fastest, or 0 where the per-layer launches are faster.  Microseconds, fitted
// to depths 2 .. 8 and 1 .. 16 images of 8 to 1000 pixels a side: 1.4 + 0.45
// per row and pipeline step for each round of 256 workgroups (0.28 at depth 2,
// 0.69 from depth 7, where two hidden layers share a SIMD), against 3.9 per
// launch and 0.031 + 0.034 per hidden layer for every thousand pixels.  Depth
// 5: 1 x 320 x 320 30 against 46 us, 16 x 320 x 320 186 against 255; 1024 x 8
// x 8 (a third of each strip used, four rounds) 62 against 41; depth 2, 16 x
// 320 x 320 118 against 72; depth 8, 16 x 320 x 320 516 against 420.  Where it
// takes the slower way: depth 3, 1 x 1000 x 1000 85 against 80; depth 8, 16 x 320
// x 320 in strips of 81 rows 440 against 409.
int cnn_net_rows(int depth, int n, int h, int w);
void cnn_net(hipStream_t st, const CnnLayer* ls, int depth, const float* x, float* y, int n, int h, int w, int rows);
// The last layer of a training pass: y = conv(in) + b is not stored but
// compared with t: the loss 1/(2m) sum (y - t)^2 over the m = 6 n h w outputs
// as cnn_mse_blocks fp64 partial sums, and dz = (y - t) / m in bf16, padded to
// 8 channels.
void cnn_conv_last_mse(hipStream_t st, const void* in, const void* wk, const float* b, const float* t, void* dz,
                       double* part, int n, int h, int w);
int cnn_mse_blocks(int n, int h, int w);
// din = (conv^T dz) * [act > 0], bf16, of a layer 32 -> cout.
void cnn_conv_backward_data(hipStream_t st, int cout, const void* dz, const void* wt, const void* act, void* din, int n,
                            int h, int w);
// Per-block partial gradients of a layer (in: bf16, fp32 for the first), and
// their sums in every layer's g.
size_t cnn_wgrad_part_floats(int cin, int cout, int n, int h, int w);
void cnn_conv_wgrad(hipStream_t st, CnnLayer& L, const void* in, const void* dz, int n, int h, int w);
void cnn_reduce_grads(hipStream_t st, const CnnLayer* ls, int count);
// One Adam update; c1 = 1 - b1^t, c2 = 1 - b2^t.
void cnn_adam(hipStream_t st, float* w, const float* g, float* m, float* v, int64_t n, float lr, float b1, float b2,
              float eps, float c1, float c2);
// Warm start from a complex64 image u0 (n pixels); ss points to the sum of
// |u0|^2 on the device, from which the input scale RMS(u0) is taken.
void cnn_ws_pack(hipStream_t st, const void* u0, int64_t n, const double* ss, float* x);
void cnn_ws_unpack(hipStream_t st, const float* x, const float* y, int64_t n, const double* ss, void* u, void* v);

}  // namespace pdt
