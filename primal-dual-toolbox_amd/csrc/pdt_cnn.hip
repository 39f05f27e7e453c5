// pdt_cnn.hip -- the warm-start network: conv3x3 layers (zero padding,
// stride 1) with ReLU between them, as implicit GEMMs on the bf16 MFMA
// (v_mfma_f32_16x16x32_bf16, fp32 accumulation), its backward pass, an MSE
// loss and Adam.
//
// Layout: activations NHWC (channel fastest), bf16 between layers (the
// 6-channel output gradient padded to 8), fp32 at the input and output.
// Master parameters fp32, per layer W[tap][co][ci] (tap = 3 ky + kx) then
// b[co]; the MFMA takes bf16 copies in the order its lanes load them
// (pack_weights).
//
// MFMA operand layout (v_mfma_f32_16x16x32_bf16, wave64): lane l holds
// A[l % 16][(l / 16) * 8 + i] and B[(l / 16) * 8 + i][l % 16], i < 8, and
// receives C[(l / 16) * 4 + i][l % 16], i < 4.
//
// The convolutions put output channels on the A rows and 16 neighbouring
// pixels of a row on the B columns: a lane then reads 8 consecutive channels
// of one pixel (the wave 1 KB of contiguous memory) and, with the two
// 16-channel tiles interleaved (tile t, row 4 g + i holds channel
// 8 g + 4 t + i), receives 8 consecutive channels of one pixel.  No operand
// or result passes through LDS.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "pdt_cnn.hpp"
#include "pdt_pixel.hpp"

namespace pdt {

namespace {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f16 __attribute__((ext_vector_type(16)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));
// two floats at 4-byte alignment (the caller's arrays)
struct __attribute__((packed, aligned(4))) F2 {
  float a, b;
};

constexpr int kConvThreads = 256;  // 4 waves, each on its own strips

__device__ __forceinline__ f4 mfma(const bf8& a, const bf8& b, const f4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f16 mfma(const bf8& a, const bf8& b, const f16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// v where m is all ones, 0 where it is 0
__device__ __forceinline__ bf8 keep(bf8 v, uint32_t m) {
  u4 x = __builtin_bit_cast(u4, v);
  x &= m;
  return __builtin_bit_cast(bf8, x);
}

// Input channels as the kernels see them (the 6-channel gradient as 8), the
// 32-wide k-steps and the 16-wide output-channel tiles of a convolution.
__host__ __device__ constexpr int chan_in(int cin) { return cin == 6 ? 8 : cin; }
__host__ __device__ constexpr int ksteps(int cin) { return (9 * chan_in(cin) + 31) / 32; }
__host__ __device__ constexpr int tiles_out(int cout) { return (cout + 15) / 16; }
// Output channel of row m of tile t.
__host__ __device__ constexpr int row_channel(int nt, int t, int m) { return nt == 2 ? (m >> 2) * 8 + t * 4 + (m & 3) : m; }

// Epilogues of the convolutions.
enum { EPI_RELU_BF16 = 0, EPI_F32 = 1, EPI_MASK_BF16 = 2, EPI_MSE = 3 };

// The rows of all strip columns (n images, ns strips of 16 or 32 pixels, h
// rows) in equal contiguous shares, one per wave: with as many waves as stay
// resident, no last round of a few waves.
// (32-bit: 2^32 rows of 16 pixels would be 4 TB of activations.)
struct Share {
  uint32_t a, b;
};
__device__ __forceinline__ uint32_t strip_rows(int n, int h, int w, int width) {
  return uint32_t(n) * uint32_t(h) * uint32_t((w + width - 1) / width);
}
template <int WAVES>
__device__ __forceinline__ Share share_of(uint32_t rows) {
  const uint32_t nw = gridDim.x * WAVES, q = rows / nw, r = rows - q * nw;
  // (neighbouring strips and rows, which share input rows, to one XCD and its L2)
  const uint32_t id = uint32_t(xcd_item(blockIdx.x, gridDim.x)) * WAVES + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t a = id * q + min(id, r);
  return {a, a + q + (id < r ? 1u : 0u)};
}
// The next piece of a share: rows [y0, y1) of the strip from x0 of image img.
struct Piece {
  int img, x0, y0, y1;
};
template <int WIDTH>
__device__ __forceinline__ Piece next_piece(Share& s, int h, int w) {
  const uint32_t ns = (w + WIDTH - 1) / WIDTH, col = s.a / uint32_t(h), y0 = s.a - col * h;
  const uint32_t y1 = min(uint32_t(h), y0 + (s.b - s.a)), img = col / ns;
  s.a += y1 - y0;
  return {int(img), int(col - img * ns) * WIDTH, int(y0), int(y1)};
}

// Blocks of a convolution: at least 4 rows of 16 pixels per wave, and no more
// waves than stay resident (2 or 8 per SIMD).
int conv_blocks(int n, int h, int w, int waves_per_simd) {
  const int64_t b = (int64_t(n) * h * ((w + 15) / 16) + 15) / 16;
  return int(b < 256 * waves_per_simd ? b : 256 * waves_per_simd);
}

// What the epilogue of a pixel reads besides the sums, loaded rows ahead:
// the 8 channels of the mask (EPI_MASK_BF16) or the 4 (lane group 0) or 2
// (group 1) targets (EPI_MSE).
template <int EPI> struct Aux {};
template <> struct Aux<EPI_MASK_BF16> {
  bf8 a;
};
template <> struct Aux<EPI_MSE> {
  F2 a, b;
};
// p: pixel index of a lane inside the image (lanes past it pass its last column)
template <int EPI>
__device__ __forceinline__ Aux<EPI> load_aux(const void* aux, size_t p) {
  const int g = (threadIdx.x & 63) >> 4;
  if constexpr (EPI == EPI_MASK_BF16) {
    return {*reinterpret_cast<const bf8*>(static_cast<const __bf16*>(aux) + p * 32 + g * 8)};
  } else if constexpr (EPI == EPI_MSE) {
    const float* t = static_cast<const float*>(aux) + p * 6;  // groups 2 and 3 hold no channel
    return {*reinterpret_cast<const F2*>(t + (g == 1 ? 4 : 0)), *reinterpret_cast<const F2*>(t + 2)};
  } else {
    return {};
  }
}

// Bias, ReLU or mask, and the stores of one row of 16 pixels: acc[t][i] is
// channel row_channel(T, t, 4 (lane / 16) + i) of pixel p (in: a lane of the
// image's columns).  EPI_MSE: dz = (y - t) / M in bf16 and sum (y - t)^2.
template <int T, int EPI>
__device__ __forceinline__ void conv_store(const f4 (&acc)[T], const float (&b)[4 * T], size_t p, bool in, void* out,
                                           const Aux<EPI>& aux, float m, double& ss) {
  const int g = (threadIdx.x & 63) >> 4;
  if constexpr (EPI == EPI_RELU_BF16 || EPI == EPI_MASK_BF16) {
    static_assert(T == 2, "8 channels per lane");
    bf8 o;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      if constexpr (EPI == EPI_RELU_BF16) o[c] = __bf16(fmaxf(acc[c / 4][c % 4] + b[c], 0.f));
      else o[c] = __bf16(float(aux.a[c]) > 0.f ? acc[c / 4][c % 4] : 0.f);
    }
    if (in) *reinterpret_cast<bf8*>(static_cast<__bf16*>(out) + p * 32 + g * 8) = o;
  } else {
    // 6 channels: lanes of group 0 hold 0..3, of group 1 hold 4 and 5
    if (!in || g > 1) return;
    const float v0 = acc[0][0] + b[0], v1 = acc[0][1] + b[1], v2 = acc[0][2] + b[2], v3 = acc[0][3] + b[3];
    if constexpr (EPI == EPI_F32) {
      F2* y = reinterpret_cast<F2*>(static_cast<float*>(out) + p * 6 + g * 4);
      y[0] = {v0, v1};
      if (g == 0) y[1] = {v2, v3};
    } else {
      const float d0 = v0 - aux.a.a, d1 = v1 - aux.a.b, d2 = g == 0 ? v2 - aux.b.a : 0.f, d3 = g == 0 ? v3 - aux.b.b : 0.f;
      ss += double(d0) * d0 + double(d1) * d1;
      ss += double(d2) * d2 + double(d3) * d3;
      const bf4 z = {__bf16(d0 / m), __bf16(d1 / m), __bf16(d2 / m), __bf16(d3 / m)};
      *reinterpret_cast<bf4*>(static_cast<__bf16*>(out) + p * 8 + g * 4) = z;
    }
  }
}

// The loss partial of a block (EPI_MSE), summed in a fixed order.
__device__ __forceinline__ void store_loss(double ss, double* lpart) {
  __shared__ double red[4];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) ss += __shfl_down(ss, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  if (threadIdx.x == 0) lpart[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// 32 input channels.  A wave walks down its strip holding the weights of all
// nine taps and the sums of three output rows in registers: the three
// fragments of an input row (dx = -1, 0, 1; 16 pixels x 32 channels each,
// loaded one row ahead) serve the output rows above, at and below it, so
// each is read once per strip and not once per tap row.  What bounds it is
// memory (64 bytes in and 64 out per pixel against 9216 products).  The taps
// of a pixel are summed in order 0..8.
// 16 x 320 x 320, 32 -> 32: 50 us forward, 57 us backward-data (4.2 and 5.5
// TB/s on 210 and 315 MB; counted 252 and 371 MB, 5.0 and 6.5 TB/s, with the
// matrix cores busy 13 us); 163 and 233 us with a wave per 64 pixels, nine
// fragment loads per 16 pixels and results through LDS.  Rows one step ahead
// instead of three: 75 and 104 us; shares of 16 rows instead of equal ones (a
// last round of few waves): 57.6 and 67.4 us.
template <int T, int EPI>
__global__ __launch_bounds__(kConvThreads) void conv32_kernel(const __bf16* __restrict__ in, const bf8* __restrict__ wk,
                                                              const float* __restrict__ bias, void* out,
                                                              const void* __restrict__ aux, double* lpart, int n, int h,
                                                              int w) {
  const int lane = threadIdx.x & 63, g = lane >> 4;
  double ss = 0;
  bf8 wt[9][T];
#pragma unroll
  for (int k = 0; k < 9; ++k)
#pragma unroll
    for (int t = 0; t < T; ++t) wt[k][t] = wk[(k * T + t) * 64 + lane];
  float b[4 * T];
#pragma unroll
  for (int c = 0; c < 4 * T; ++c) {
    const int ch = T == 2 ? g * 8 + c : g * 4 + c;
    b[c] = bias && (T == 2 || ch < 6) ? bias[ch] : 0.f;
  }
  const float m = EPI == EPI_MSE ? float(int64_t(n) * h * w * 6) : 0.f;
  Share sh = share_of<4>(strip_rows(n, h, w, 16));
  while (sh.a < sh.b) {
    const Piece s = next_piece<16>(sh, h, w);
    const int x = s.x0 + (lane & 15);
    int off[3];
    uint32_t ok[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const int xx = x + d - 1;
      ok[d] = xx >= 0 && xx < w ? ~0u : 0u;
      off[d] = min(max(xx, 0), w - 1) * 32 + g * 8;
    }
    const size_t base = size_t(s.img) * h;
    // Input rows are loaded three steps ahead, into the registers of the row
    // just used (and the epilogue's operands of the row it completes with
    // them), without branches (clamped rows and columns, masked at use), so
    // that the waits count them exactly: two rows per step stay in flight.
    struct Row {
      bf8 f[3];
      Aux<EPI> aux;
    };
    auto load = [&](Row& r, int yi) {
      const __bf16* row = in + (base + min(max(yi, 0), h - 1)) * size_t(w) * 32;
#pragma unroll
      for (int d = 0; d < 3; ++d) r.f[d] = *reinterpret_cast<const bf8*>(row + off[d]);
      r.aux = load_aux<EPI>(aux, (base + min(max(yi - 1, 0), h - 1)) * w + min(x, w - 1));
    };
    // input row yi for the output rows yi + 1 (first: its sums start here),
    // yi and yi - 1 (last: done)
    auto step = [&](int yi, Row& r, f4 (&first)[T], f4 (&mid)[T], f4 (&last)[T]) {
      const uint32_t inside = yi >= 0 && yi < h ? ~0u : 0u;
#pragma unroll
      for (int t = 0; t < T; ++t) first[t] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const bf8 c = keep(r.f[d], ok[d] & inside);
#pragma unroll
        for (int t = 0; t < T; ++t) {
          first[t] = mfma(wt[d][t], c, first[t]);
          mid[t] = mfma(wt[3 + d][t], c, mid[t]);
          last[t] = mfma(wt[6 + d][t], c, last[t]);
        }
      }
      const Aux<EPI> ax = r.aux;
      load(r, yi + 3);
      const int yo = yi - 1;
      if (yo >= s.y0 && yo < s.y1) conv_store<T, EPI>(last, b, (base + yo) * w + x, x < w, out, ax, m, ss);
    };
    f4 r0[T], r1[T], r2[T];
#pragma unroll
    for (int t = 0; t < T; ++t) r0[t] = r1[t] = r2[t] = f4{0.f, 0.f, 0.f, 0.f};
    Row a, c, e;
    load(a, s.y0 - 1);
    load(c, s.y0);
    load(e, s.y0 + 1);
    for (int yi = s.y0 - 1; yi <= s.y1; yi += 3) {
      step(yi, a, r0, r1, r2);
      step(yi + 1, c, r2, r0, r1);
      step(yi + 2, e, r1, r2, r0);
    }
  }
  if constexpr (EPI == EPI_MSE) store_loss(ss, lpart);
}

// First layer, 2 input channels in fp32: k = 2 tap + channel fills 18 of one
// 32-wide k-step; lane group g takes the pixels of taps 4 g .. 4 g + 3 (8
// bytes each), rounded to bf16.  Bound by its 64-byte output per pixel.
// 16 x 320 x 320: 33 us (88 us, and 8 us for a separate conversion to bf16,
// with single-value gathers).
__global__ __launch_bounds__(kConvThreads) void conv_in_kernel(const float* __restrict__ in, const bf8* __restrict__ wk,
                                                               const float* __restrict__ bias, __bf16* out, int n, int h,
                                                               int w) {
  const int lane = threadIdx.x & 63, g = lane >> 4;
  const bf8 w0 = wk[lane], w1 = wk[64 + lane];
  float b[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) b[c] = bias[g * 8 + c];
  double ss = 0;
  Share sh = share_of<4>(strip_rows(n, h, w, 16));
  while (sh.a < sh.b) {
    const Piece s = next_piece<16>(sh, h, w);
    const int x = s.x0 + (lane & 15);
    const size_t base = size_t(s.img) * h;
#pragma unroll 2
    for (int y = s.y0; y < s.y1; ++y) {
      bf8 f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int tap = 4 * g + j, yy = y + tap / 3 - 1, xx = x + tap % 3 - 1;
        F2 v = {0.f, 0.f};
        if (tap < 9 && yy >= 0 && yy < h && xx >= 0 && xx < w)
          v = *reinterpret_cast<const F2*>(in + 2 * ((base + yy) * w + xx));
        f[2 * j] = __bf16(v.a);
        f[2 * j + 1] = __bf16(v.b);
      }
      const f4 z = {0.f, 0.f, 0.f, 0.f};
      const f4 acc[2] = {mfma(w0, f, z), mfma(w1, f, z)};
      conv_store<2, EPI_RELU_BF16>(acc, b, (base + y) * w + x, x < w, out, Aux<EPI_RELU_BF16>{}, 0.f, ss);
    }
  }
}

// Backward-data pass of the last layer: its 6-channel gradient, padded to 8,
// against the flipped weights: lane group g of k-step s takes the 8 channels
// of tap 4 s + g (16 bytes of one pixel).  Memory-bound: 16 x 320 x 320 in
// 40 us, 5.9 TB/s on 236 MB (179 us with the channels gathered one by one).
__global__ __launch_bounds__(kConvThreads) void conv8_kernel(const __bf16* __restrict__ dz, const bf8* __restrict__ wk,
                                                             __bf16* out, const __bf16* __restrict__ act, int n, int h,
                                                             int w) {
  const int lane = threadIdx.x & 63, g = lane >> 4;
  bf8 wt[3][2];
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int t = 0; t < 2; ++t) wt[k][t] = wk[(k * 2 + t) * 64 + lane];
  const float b[8] = {};
  double ss = 0;
  Share sh = share_of<4>(strip_rows(n, h, w, 16));
  while (sh.a < sh.b) {
    const Piece s = next_piece<16>(sh, h, w);
    const int x = s.x0 + (lane & 15);
    const size_t base = size_t(s.img) * h;
#pragma unroll 2
    for (int y = s.y0; y < s.y1; ++y) {
      f4 acc[2] = {f4{0.f, 0.f, 0.f, 0.f}, f4{0.f, 0.f, 0.f, 0.f}};
      const Aux<EPI_MASK_BF16> ax = load_aux<EPI_MASK_BF16>(act, (base + y) * w + min(x, w - 1));
      bf8 f[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const int tap = 4 * k + g, yy = y + tap / 3 - 1, xx = x + tap % 3 - 1;
        const bool ok = tap < 9 && yy >= 0 && yy < h && xx >= 0 && xx < w;
        const bf8 v = *reinterpret_cast<const bf8*>(dz + (ok ? (base + yy) * w + xx : (base + y) * w) * 8);
        f[k] = keep(v, ok ? ~0u : 0u);
      }
#pragma unroll
      for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[t] = mfma(wt[k][t], f[k], acc[t]);
      conv_store<2, EPI_MASK_BF16>(acc, b, (base + y) * w + x, x < w, out, ax, 0.f, ss);
    }
  }
}

// ---------------------------------------------------------------------------
// The whole network on a strip (inference): a workgroup has one wave per
// layer, and rows of activations go from wave to wave through LDS.  At step t
// wave l takes the row that wave l - 1 wrote at step t - 1 (32 pixels x 32
// channels), adds it to the sums of the three output rows that it touches, and
// writes the row it completes; the first wave gathers the input, the last one
// stores the output.  One barrier a step.  The weights of a layer stay in its
// wave's registers.  Of the 32 columns one on each side is lost per layer
// after the first, of the rows as many above and below, and the pipeline takes
// two steps a layer to fill.  Activations outside the image are zero, as the
// layers' zero padding has them, and the products are added in the order of
// the per-layer kernels: the outputs are the same bits.
// Bound by a hidden wave's chain: 18 matrix instructions (576 clocks), the LDS
// round trip, the rounding and the barrier, 0.45 us a step (0.60 us with
// 16 x 16 tiles and taps gathered from memory).  Depth 5, a call: 1 x 320 x
// 320 30 us (46 in five launches), 4 x 320 x 320 61 (84), 16 x 320 x 320 186
// (255).
// ---------------------------------------------------------------------------
constexpr int kNetCols = 32;        // columns of a strip, halo included
constexpr int kNetPix = kNetCols + 2;  // a staged row has one unused pixel on either side
constexpr int kNetBlocks = 256;     // workgroups at a time: one per compute unit (registers)
constexpr int kNetLayers = 8;       // deepest network (its halo leaves 18 columns)

// LDS slot (8 channels each) of chunk c of staged pixel p: any 16 neighbouring
// pixels' chunks c lie on different banks.
__device__ __forceinline__ int net_slot(int p, int c) { return p * 4 + (c ^ ((p >> 2) & 3)); }

// Steps of a workgroup that stores R rows, a multiple of three.
__host__ __device__ constexpr int net_steps(int R, int depth) { return (R + 3 * (depth - 1) + 2) / 3 * 3; }

// The first layer: its rows to `next`.  One load per input row (a pixel per
// lane), six rows ahead, rounded to bf16 into a ring of three rows in LDS; a
// lane gathers its taps 4 g .. 4 g + 3 (k = 2 tap + channel) from there, those
// past the ninth from a cell that holds zero.
__device__ __forceinline__ void net_first(const bf8* wk, const float* bias, const float* in, bf8* next, uint32_t* taps,
                                          int steps, size_t base, int ya, int h, int xr, int w) {
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const bf8 w0 = wk[lane], w1 = wk[64 + lane];
  float b[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) b[i] = bias[g * 8 + i];
  const int xl = xr - 1 + lane, xc = min(max(xl, 0), w - 1);
  const bool in_cols = lane < kNetPix && xl >= 0 && xl < w;
  if (lane == 0) taps[3 * kNetPix] = 0;
  auto load = [&](F2& q, int yr) {
    q = *reinterpret_cast<const F2*>(in + 2 * ((base + min(max(yr, 0), h - 1)) * w + xc));
  };
  auto stage = [&](F2 q, int yr, int slot) {
    asm volatile("" : "+v"(q.a), "+v"(q.b));  // not rounded, hence not waited for, before its step
    const bool ok = in_cols && yr >= 0 && yr < h;
    typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
    const bf2 v = {__bf16(ok ? q.a : 0.f), __bf16(ok ? q.b : 0.f)};
    if (lane < kNetPix) taps[slot * kNetPix + lane] = __builtin_bit_cast(uint32_t, v);
  };
  // cells of the taps for row slot (0, 1, 2) of the output row
  int cell[3][4], step2[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int tap = 4 * g + j;
#pragma unroll
    for (int k = 0; k < 3; ++k) cell[k][j] = tap < 9 ? (k + 2 + tap / 3) % 3 * kNetPix + c + tap % 3 : 3 * kNetPix;
    step2[j] = tap < 9 ? 16 : 0;
  }
  // row ya + t in slot t % 3 (t counted from -1 as 2)
  auto step = [&](int t, int k, F2& q) {
    const int yr = ya + t;
    stage(q, yr + 1, (k + 1) % 3);
    load(q, yr + 7);
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const int x = xr + m * 16 + c;
      u4 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = taps[cell[k][j] + m * step2[j]];
      const bf8 f = __builtin_bit_cast(bf8, v);
      const f4 z = {0.f, 0.f, 0.f, 0.f};
      const f4 acc[2] = {mfma(w0, f, z), mfma(w1, f, z)};
      bf8 o;
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] = __bf16(fmaxf(acc[i / 4][i % 4] + b[i], 0.f));
      next[(t & 1) * (kNetPix * 4) + net_slot(m * 16 + c + 1, g)] =
          keep(o, yr >= 0 && yr < h && x >= 0 && x < w ? ~0u : 0u);
    }
    wg_barrier();
  };
  F2 p, q, r[6];
  load(p, ya - 1);
  load(q, ya);
#pragma unroll
  for (int i = 0; i < 6; ++i) load(r[i], ya + 1 + i);
  stage(p, ya - 1, 2);
  stage(q, ya, 0);
  for (int t = 0; t < steps; t += 3) {
    step(t, 0, r[0]);
    step(t + 1, 1, r[1]);
    step(t + 2, 2, r[2]);
    if ((t += 3) >= steps) break;
    step(t, 0, r[3]);
    step(t + 1, 1, r[4]);
    step(t + 2, 2, r[5]);
  }
}

// A hidden layer: its rows to `next`.  32 x 32 matrix tiles, channels by
// pixels: half the instructions of 16 x 16 tiles, which one wave per SIMD does
// not issue back to back (28 clocks each instead of 16; 32 clocks of 32 here).
__device__ __forceinline__ void net_hidden(const bf8* wk, const float* bias, const bf8* prev, bf8* next, int l,
                                           int steps, int ya, int h, int xr, int w) {
  const int lane = threadIdx.x & 63, half = lane >> 5, c = lane & 31;
  // Row c of the tile is the output channel that leaves a lane with channels
  // 16 half .. 16 half + 15 of its pixel.
  const int ch = 16 * ((c >> 2) & 1) + 4 * (c >> 3) + (c & 3);
  bf8 wt[9][2];
#pragma unroll
  for (int k = 0; k < 9; ++k)
#pragma unroll
    for (int s = 0; s < 2; ++s)
      wt[k][s] = wk[(k * 2 + ((ch >> 2) & 1)) * 64 + (2 * s + half) * 16 + (ch >> 3) * 4 + (ch & 3)];
  float b[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) b[i] = bias[16 * half + i];
  f16 r0, r1, r2;
#pragma unroll
  for (int i = 0; i < 16; ++i) r0[i] = r1[i] = r2[i] = 0.f;
  const int x = xr + c;
  const bool in_cols = x >= 0 && x < w;
  auto step = [&](int t, f16& first, f16& mid, f16& last) {
    const bf8* in = prev + ((t - 1) & 1) * (kNetPix * 4);
    bf8 f[3][2];
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int s = 0; s < 2; ++s) f[d][s] = in[net_slot(c + d, 2 * s + half)];
#pragma unroll
    for (int i = 0; i < 16; ++i) first[i] = 0.f;
    // The row that is completed runs ahead, so that its bias, rounding and
    // store are beside the products of the other two.
#pragma unroll
    for (int j = 0; j < 6; ++j) {
      last = mfma(wt[6 + j / 2][j & 1], f[j / 2][j & 1], last);
      const int k = j >> 1;
      if (j & 1)
        first = mfma(wt[k / 2][k & 1], f[k / 2][k & 1], first);
      else
        mid = mfma(wt[3 + k / 2][k & 1], f[k / 2][k & 1], mid);
    }
#pragma unroll
    for (int k = 3; k < 6; ++k) {
      mid = mfma(wt[3 + k / 2][k & 1], f[k / 2][k & 1], mid);
      first = mfma(wt[k / 2][k & 1], f[k / 2][k & 1], first);
    }
    const int yo = ya + t - 2 * l;
    const unsigned mask = yo >= 0 && yo < h && in_cols ? ~0u : 0u;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      bf8 o;
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] = __bf16(fmaxf(last[8 * q + i] + b[8 * q + i], 0.f));
      next[(t & 1) * (kNetPix * 4) + net_slot(c + 1, 2 * half + q)] = keep(o, mask);
    }
    wg_barrier();
  };
  for (int t = 0; t < steps; t += 3) {
    step(t, r0, r1, r2);
    step(t + 1, r2, r0, r1);
    step(t + 2, r1, r2, r0);
  }
}

// The last layer: rows [y0, y1) and columns [s0, s1) to y.
__device__ __forceinline__ void net_last(const bf8* wk, const float* bias, const bf8* prev, float* y, int l, int steps,
                                         size_t base, int ya, int y0, int y1, int xr, int s0, int s1, int w) {
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  bf8 wt[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) wt[k] = wk[k * 64 + lane];
  float b[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) b[i] = g * 4 + i < 6 ? bias[g * 4 + i] : 0.f;
  f4 r0[2][1], r1[2][1], r2[2][1];
#pragma unroll
  for (int m = 0; m < 2; ++m) r0[m][0] = r1[m][0] = r2[m][0] = f4{0.f, 0.f, 0.f, 0.f};
  auto step = [&](int t, f4 (&first)[2][1], f4 (&mid)[2][1], f4 (&last)[2][1]) {
    const bf8* in = prev + ((t - 1) & 1) * (kNetPix * 4);
    bf8 f[3][2];
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int m = 0; m < 2; ++m) f[d][m] = in[net_slot(m * 16 + c + d, g)];
    first[0][0] = first[1][0] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        last[m][0] = mfma(wt[6 + d], f[d][m], last[m][0]);
        first[m][0] = mfma(wt[d], f[d][m], first[m][0]);
        mid[m][0] = mfma(wt[3 + d], f[d][m], mid[m][0]);
      }
    const int yo = ya + t - 2 * l;
    if (yo >= y0 && yo < y1)
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const int x = xr + m * 16 + c;
        double ss = 0;
        conv_store<1, EPI_F32>(last[m], b, (base + yo) * w + x, x >= s0 && x < s1, y, Aux<EPI_F32>{}, 0.f, ss);
      }
    wg_barrier();
  };
  for (int t = 0; t < steps; t += 3) {
    step(t, r0, r1, r2);
    step(t + 1, r2, r0, r1);
    step(t + 2, r1, r2, r0);
  }
}

__global__ __launch_bounds__(64 * kNetLayers) __attribute__((amdgpu_waves_per_eu(2))) void net_kernel(
    const float* __restrict__ in, float* y, CnnLayers ls, int depth, int n, int h, int w, int R) {
  __shared__ __attribute__((aligned(16))) bf8 ring[(kNetLayers - 1) * 2 * kNetPix * 4];
  __shared__ uint32_t taps[3 * kNetPix + 1];
  const int halo = depth - 1, ow = kNetCols - 2 * halo, ns = (w + ow - 1) / ow, nc = (h + R - 1) / R;
  const int id = xcd_item(blockIdx.x, gridDim.x), img = id / (ns * nc), r = id - img * ns * nc, cy = r / ns;
  const int s0 = (r - cy * ns) * ow, s1 = min(w, s0 + ow), xr = s0 - halo;
  const int y0 = cy * R, y1 = min(h, y0 + R), ya = y0 - halo;
  const size_t base = size_t(img) * h;
  const int steps = net_steps(R, depth);
  const int l = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const CnnLayer& L = ls.l[l];
  const bf8* wk = static_cast<const bf8*>(L.wk);
  const float* bias = L.w + 9 * L.cin * L.cout;
  const bf8* prev = ring + (l - 1) * 2 * (kNetPix * 4);
  bf8* next = ring + l * 2 * (kNetPix * 4);
  if (l == depth - 1) {
    net_last(wk, bias, prev, y, l, steps, base, ya, y0, y1, xr, s0, s1, w);
  } else if (l > 0) {
    net_hidden(wk, bias, prev, next, l, steps, ya, h, xr, w);
  } else {
    net_first(wk, bias, in, next, taps, steps, base, ya, h, xr, w);
  }
}

// ---------------------------------------------------------------------------
// Weight gradient: dW[co][tap, ci] = sum_p dz[p][co] in[p + off(tap)][ci],
// the pixels on the k axis.  Both operands are stored pixel by pixel, so a
// lane, which needs 8 pixels of one channel, gets them from LDS through
// ds_read_b64_tr_b16: of a 16-lane group, lane i names 4 channels of row
// i / 4 and receives channel i of the 4 rows.  A wave walks down strips of 32
// pixels: the gradient fragments of three rows stay in registers, the
// fragments of an input row (3 dx x 32 channels) pair with all three, and the
// sums of all taps (32 x 288 values) stay in its accumulators to the end of
// its rows.  Waves stage their own rows, so no barrier separates them.
// ---------------------------------------------------------------------------
constexpr int kGradWaves = 8, kGradThreads = 64 * kGradWaves, kGradStrip = 32;
constexpr int kGradBlocks = 256;  // one per CU

#define PDT_WAVE_FENCE() __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront")

// LDS slot of 4-channel chunk c (0..CH/4) of staged pixel p, rows of CH
// channels: of 32 channels, the two 32-byte halves trade places every 8
// pixels, so that the 8-byte reads of lane groups 8 pixels apart fall on
// different banks.
template <int CH>
__device__ __forceinline__ int grad_slot(int p, int c) {
  return p * (CH / 4) + (CH == 32 ? (c ^ (((p >> 3) & 1) << 2)) : c);
}
// 8 pixels (from p, one per k) of channel c0 + lane % 16 for each lane group.
template <int CH>
__device__ __forceinline__ bf8 grad_frag(const bf4* s, int p, int c0) {
  const int lane = threadIdx.x & 63, i = lane & 15, r = p + (lane >> 4) * 8 + (i >> 2), c = c0 / 4 + (i & 3);
  typedef __attribute__((address_space(3))) bf4 lds_bf4;
  const bf4 a = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf4*)(s + grad_slot<CH>(r, c)));
  const bf4 b = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf4*)(s + grad_slot<CH>(r + 4, c)));
  return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}

// Channels of a staged gradient pixel: 32, or 16 for the padded 6-channel one
// (8 stored, 8 zero).
__host__ __device__ constexpr int grad_ch(int cout) { return cout == 32 ? 32 : 16; }

// Adds the accumulators of the block's waves in wave order and writes the
// block's partial, [tile][lane][i] then db[co]; sum is the block's LDS.  (The
// barrier is at the head of a loop whose last LDS store is at its end:
// wg_barrier, whose wait does not depend on the loop being unrolled.)
template <int NT, int CT>
__device__ __forceinline__ void grad_partial(const f4 (&acc)[NT], const f4 (&db)[CT], float* sum, float* part) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  f4* s4 = reinterpret_cast<f4*>(sum);
  for (int q = 0; q < kGradWaves; ++q) {
    wg_barrier();
    if (wave == q) {
#pragma unroll
      for (int t = 0; t < NT; ++t) s4[t * 64 + lane] = q ? s4[t * 64 + lane] + acc[t] : acc[t];
      // db: every column of the product with ones holds the same sums
#pragma unroll
      for (int t = 0; t < CT; ++t)
        if ((lane & 15) == 0) {
          f4* d = s4 + NT * 64 + t * 4 + (lane >> 4);
          *d = q ? *d + db[t] : db[t];
        }
    }
  }
  wg_barrier();
  constexpr int N4 = NT * 64 + CT * 4;
  f4* o = reinterpret_cast<f4*>(part) + size_t(blockIdx.x) * N4;
  for (int e = threadIdx.x; e < N4; e += kGradThreads) o[e] = s4[e];
}

// 32 input channels; COUT 32, or 6 with dz padded to 8 channels.
// 16 x 320 x 320, 32 -> 32: 60 us for 210 MB of operands, of which the strips'
// overlapping borders make 283 MB of traffic, 4.7 TB/s; the matrix cores are
// busy 13 us of it.  (476 us with single 2-byte LDS reads and 1024 partials.)
template <int COUT>
__global__ __launch_bounds__(kGradThreads) void wgrad32_kernel(const __bf16* __restrict__ in,
                                                               const __bf16* __restrict__ dz, float* part, int n, int h,
                                                               int w) {
  constexpr int CT = tiles_out(COUT), NT = 9 * CT * 2, DC = grad_ch(COUT), DS = COUT == 32 ? 32 : 8;
  constexpr int IPX = kGradStrip + 2;                             // staged input pixels
  constexpr int IN4 = (IPX + 6) * 8, DZ4 = kGradStrip * (DC / 4);  // 4-channel slots (input rows end on a multiple of 8 pixels)
  constexpr int STAGE = 2 * (IN4 + DZ4);
  constexpr int SUM4 = NT * 64 + CT * 4;  // f4 of the partial
  constexpr size_t kLds = size_t(kGradWaves) * STAGE * 8 > size_t(SUM4) * 16 ? size_t(kGradWaves) * STAGE * 8 : size_t(SUM4) * 16;
  __shared__ __attribute__((aligned(16))) char smem[kLds];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  bf4* const stage = reinterpret_cast<bf4*>(smem) + wave * STAGE;
  f4 acc[NT], db[CT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < CT; ++t) db[t] = f4{0.f, 0.f, 0.f, 0.f};
  bf8 ones, zero;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    ones[i] = __bf16(1.f);
    zero[i] = __bf16(0.f);
  }
  if (COUT != 32)  // the upper 8 channels of the padded gradient stay zero
    for (int q = 0; q < 2; ++q)
      if (lane < kGradStrip) *reinterpret_cast<bf8*>(stage + q * (IN4 + DZ4) + IN4 + lane * 4 + 2) = zero;
  Share sh = share_of<kGradWaves>(strip_rows(n, h, w, kGradStrip));
  while (sh.a < sh.b) {
    const Piece pc = next_piece<kGradStrip>(sh, h, w);
    const int x0 = pc.x0, y0 = pc.y0, y1 = pc.y1;
    const size_t base = size_t(pc.img) * h;
    // staging: 16-byte pieces (8 channels of a pixel); input pixels x0 - 1 ..
    // x0 + 32 as pieces lane, lane + 64 and (lanes 0..7) lane + 128
    bf8 si[3], sd[2];
    auto load = [&](int yi) {  // input row yi and gradient row yi + 1 into registers
      const bool iny = yi >= 0 && yi < h;
      const __bf16* row = in + (base + (iny ? yi : 0)) * size_t(w) * 32;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const int e = lane + 64 * k, xx = x0 - 1 + (e >> 2);
        const bool ok = iny && xx >= 0 && xx < w && e < IPX * 4;
        si[k] = keep(*reinterpret_cast<const bf8*>(row + min(max(xx, 0), w - 1) * 32 + (e & 3) * 8), ok ? ~0u : 0u);
      }
      const bool dy = yi + 1 >= y0 && yi + 1 < y1;
      const __bf16* drow = dz + (base + (dy ? yi + 1 : y0)) * size_t(w) * DS;
      if constexpr (COUT == 32) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const int e = lane + 64 * k, xx = x0 + (e >> 2);
          sd[k] = keep(*reinterpret_cast<const bf8*>(drow + min(xx, w - 1) * 32 + (e & 3) * 8), dy && xx < w ? ~0u : 0u);
        }
      } else {
        const int xx = x0 + (lane & 31);
        sd[0] = keep(*reinterpret_cast<const bf8*>(drow + min(xx, w - 1) * 8), dy && xx < w ? ~0u : 0u);
      }
    };
    auto put = [&](bf4* buf) {
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const int e = lane + 64 * k;
        if (e < IPX * 4) *reinterpret_cast<bf8*>(buf + grad_slot<32>(e >> 2, (e & 3) * 2)) = si[k];
      }
      if constexpr (COUT == 32) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const int e = lane + 64 * k;
          *reinterpret_cast<bf8*>(buf + IN4 + grad_slot<32>(e >> 2, (e & 3) * 2)) = sd[k];
        }
      } else if (lane < kGradStrip) {
        *reinterpret_cast<bf8*>(buf + IN4 + lane * 4) = sd[0];
      }
    };
    // input row yi with the gradient rows yi + 1 (tap row 0, read here), yi
    // (tap row 1) and yi - 1 (tap row 2)
    bf4* cur = stage;
    bf4* nxt = stage + IN4 + DZ4;
    auto step = [&](int yi, bf8 (&a0)[CT], bf8 (&a1)[CT], bf8 (&a2)[CT]) {
      PDT_WAVE_FENCE();
      put(cur);
      PDT_WAVE_FENCE();
      if (yi < y1) load(yi + 1);
#pragma unroll
      for (int t = 0; t < CT; ++t) {
        a0[t] = grad_frag<DC>(cur + IN4, 0, t * 16);
        db[t] = mfma(a0[t], ones, db[t]);
      }
      if (yi >= 0 && yi < h) {
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            const bf8 b = grad_frag<32>(cur, d, c * 16);
#pragma unroll
            for (int t = 0; t < CT; ++t) {
              acc[((0 + d) * 2 + c) * CT + t] = mfma(a0[t], b, acc[((0 + d) * 2 + c) * CT + t]);
              acc[((3 + d) * 2 + c) * CT + t] = mfma(a1[t], b, acc[((3 + d) * 2 + c) * CT + t]);
              acc[((6 + d) * 2 + c) * CT + t] = mfma(a2[t], b, acc[((6 + d) * 2 + c) * CT + t]);
            }
          }
      }
      bf4* const sw = cur;
      cur = nxt;
      nxt = sw;
    };
    bf8 r0[CT], r1[CT], r2[CT];
#pragma unroll
    for (int t = 0; t < CT; ++t) r0[t] = r1[t] = r2[t] = zero;
    load(y0 - 1);
    for (int yi = y0 - 1; yi <= y1; yi += 3) {
      step(yi, r0, r1, r2);
      if (yi + 1 <= y1) step(yi + 1, r2, r0, r1);
      if (yi + 2 <= y1) step(yi + 2, r1, r2, r0);
    }
  }
  grad_partial<NT, CT>(acc, db, reinterpret_cast<float*>(smem), part);
}

// First layer, fp32 input of 2 channels: columns n = 2 tap + channel (18 of
// two 16-wide tiles).  The rounded input rows are staged channel by channel
// in three copies shifted by dx, so that a lane reads its 8 pixels of one
// (tap, channel) as 16 bytes.  Bound by reading dz: 16 x 320 x 320 in 32 us
// (133 us before).
__global__ __launch_bounds__(kGradThreads) void wgrad_in_kernel(const float* __restrict__ in,
                                                                const __bf16* __restrict__ dz, float* part, int n,
                                                                int h, int w) {
  constexpr int CT = 2, NT = 4;
  constexpr int ROW = 3 * 2 * kGradStrip;                // one staged input row: [dx][channel][pixel]
  constexpr int DZ4 = kGradStrip * 8;                    // gradient slots
  constexpr int STAGE = 2 * DZ4 * 8 + 3 * ROW * 2;       // bytes: two gradient rows, three input rows
  constexpr size_t kLds = size_t(kGradWaves) * STAGE;
  static_assert(kLds >= size_t(NT * 64 + CT * 4) * 16, "partial fits");
  __shared__ __attribute__((aligned(16))) char smem[kLds];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  char* const stage = smem + size_t(wave) * STAGE;
  __bf16* const sin = reinterpret_cast<__bf16*>(stage + 2 * DZ4 * 8);
  f4 acc[NT], db[CT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < CT; ++t) db[t] = f4{0.f, 0.f, 0.f, 0.f};
  bf8 ones;
#pragma unroll
  for (int i = 0; i < 8; ++i) ones[i] = __bf16(1.f);
  Share sh = share_of<kGradWaves>(strip_rows(n, h, w, kGradStrip));
  while (sh.a < sh.b) {
    const Piece pc = next_piece<kGradStrip>(sh, h, w);
    const int x0 = pc.x0, y0 = pc.y0, y1 = pc.y1;
    const size_t base = size_t(pc.img) * h;
    bf8 sd[2];
    F2 sx;
    // gradient row y and input row y + 1 into registers
    auto load_dz = [&](int y) {
      const __bf16* drow = dz + (base + y) * size_t(w) * 32;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int e = lane + 64 * k, xx = x0 + (e >> 2);
        sd[k] = keep(*reinterpret_cast<const bf8*>(drow + min(xx, w - 1) * 32 + (e & 3) * 8), xx < w ? ~0u : 0u);
      }
    };
    auto load_in = [&](int yi) {
      const int xx = x0 - 1 + lane;
      sx = {0.f, 0.f};
      if (yi >= 0 && yi < h && lane < kGradStrip + 2 && xx >= 0 && xx < w)
        sx = *reinterpret_cast<const F2*>(in + 2 * ((base + yi) * w + xx));
    };
    // staged pixel `lane` (image column x0 - 1 + lane) is pixel lane - dx of copy dx
    auto put_in = [&](int yi) {
      __bf16* r = sin + ((yi + 3) % 3) * ROW;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const int q = lane - d;
        if (q >= 0 && q < kGradStrip) {
          r[(d * 2) * kGradStrip + q] = __bf16(sx.a);
          r[(d * 2 + 1) * kGradStrip + q] = __bf16(sx.b);
        }
      }
    };
    PDT_WAVE_FENCE();
    for (int yi = y0 - 1; yi <= y0; ++yi) {
      load_in(yi);
      put_in(yi);
    }
    load_dz(y0);
    load_in(y0 + 1);
    for (int y = y0; y < y1; ++y) {
      bf4* const sz = reinterpret_cast<bf4*>(stage) + ((y - y0) & 1) * DZ4;
      PDT_WAVE_FENCE();
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int e = lane + 64 * k;
        *reinterpret_cast<bf8*>(sz + grad_slot<32>(e >> 2, (e & 3) * 2)) = sd[k];
      }
      put_in(y + 1);
      PDT_WAVE_FENCE();
      if (y + 1 < y1) {
        load_dz(y + 1);
        load_in(y + 2);
      }
      bf8 a[CT];
#pragma unroll
      for (int t = 0; t < CT; ++t) {
        a[t] = grad_frag<32>(sz, 0, t * 16);
        db[t] = mfma(a[t], ones, db[t]);
      }
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int col2 = min(c * 16 + (lane & 15), 17), tap = col2 >> 1, ci = col2 & 1;  // columns past 17: unused
        const bf8 b = *reinterpret_cast<const bf8*>(sin + ((y + tap / 3 + 2) % 3) * ROW + (tap % 3 * 2 + ci) * kGradStrip +
                                                    (lane >> 4) * 8);
#pragma unroll
        for (int t = 0; t < CT; ++t) acc[c * CT + t] = mfma(a[t], b, acc[c * CT + t]);
      }
    }
  }
  grad_partial<NT, CT>(acc, db, reinterpret_cast<float*>(smem), part);
}

// Sums the per-block partials into the master-layout gradient dW[tap][co][ci]
// and db[co].  A workgroup takes kRedOut consecutive values of the partials;
// its kRedGroups thread groups each sum every kRedGroups-th block partial, in
// block order, and the group sums are added in group order: a fixed
// summation order, so the gradient is reproducible run to run.
constexpr int kRedOut = 64, kRedGroups = 16;

// f4 of a layer's partial: 16 x 16 tiles [tap][16 input channels][16 output
// channels] (the 2-channel layer: [16 columns][16 output channels]), then db
__host__ __device__ constexpr int grad_tiles(int cin, int cout) { return (cin == 2 ? 2 : 18) * tiles_out(cout); }
__host__ __device__ constexpr int grad_floats(int cin, int cout) { return grad_tiles(cin, cout) * 256 + tiles_out(cout) * 16; }

// (every layer of the network in one launch: blockIdx.y)
__global__ __launch_bounds__(kRedOut * kRedGroups) void wgrad_reduce(CnnLayers ls) {
  __shared__ double red[kRedGroups][kRedOut];
  const CnnLayer L = ls.l[blockIdx.y];
  const int cin = L.cin, cout = L.cout, nblk = L.nblk;
  const int stride = grad_floats(cin, cout), nt = grad_tiles(cin, cout), ct = tiles_out(cout);
  if (int(blockIdx.x) * kRedOut >= stride) return;
  const int o = threadIdx.x % kRedOut, grp = threadIdx.x / kRedOut;
  const int e = blockIdx.x * kRedOut + o;
  double s = 0;
  if (e < stride) {
#pragma unroll 4
    for (int b = grp; b < nblk; b += kRedGroups) s += L.part[size_t(b) * stride + e];
  }
  red[grp][o] = s;
  __syncthreads();
  if (grp != 0 || e >= stride) return;
  double t = 0;
  for (int j = 0; j < kRedGroups; ++j) t += red[j][o];
  if (e >= nt * 256) {
    const int co = e - nt * 256;
    if (co < cout) L.g[9 * cout * cin + co] = float(t);
    return;
  }
  const int tile = e >> 8, lane = (e >> 2) & 63, co = tile % ct * 16 + (lane >> 4) * 4 + (e & 3);
  int col = lane & 15, tap;
  if (cin == 2) {
    const int n = tile / ct * 16 + col;
    tap = n >> 1;
    col = n & 1;
  } else {
    tap = tile / ct / 2;
    col += (tile / ct & 1) * 16;
  }
  if (co < cout && tap < 9) L.g[(tap * cout + co) * cin + col] = float(t);
}

// Master fp32 W[tap][co][ci] -> the bf16 operand fragments of a convolution
// with ci_n input and co_n output channels: element i of lane l of tile t of
// k-step s is the weight of output channel row_channel(t, l % 16) and k = 32 s
// + 8 (l / 16) + i, k = tap * chan_in + channel; zero where either is padding.
// back: the backward-data pass of a layer (its output channels in, its
// input channels out, taps flipped).
__device__ __forceinline__ __bf16 pack_one(const float* W, int e, int ci_n, int co_n, bool back) {
  const int nt = tiles_out(co_n), cp = chan_in(ci_n);
  const int i = e & 7, l = (e >> 3) & 63, ts = e >> 9, t = ts % nt, s = ts / nt;
  const int co = row_channel(nt, t, l & 15), k = 32 * s + 8 * (l >> 4) + i, tap = k / cp, ci = k - tap * cp;
  if (co >= co_n || tap >= 9 || ci >= ci_n) return __bf16(0.f);
  return __bf16(back ? W[((8 - tap) * ci_n + ci) * co_n + co] : W[(tap * co_n + co) * ci_n + ci]);
}
// (every layer of the network in one launch: blockIdx.y)
__global__ __launch_bounds__(256) void pack_weights(CnnLayers ls) {
  const CnnLayer L = ls.l[blockIdx.y];
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e < L.nk) static_cast<__bf16*>(L.wk)[e] = pack_one(L.w, e, L.cin, L.cout, false);
  if (L.wt && e < L.nt) static_cast<__bf16*>(L.wt)[e] = pack_one(L.w, e, L.cout, L.cin, true);
}

// Adam (Kingma & Ba, Algorithm 1) on fp32 master parameters.
__global__ __launch_bounds__(256) void adam_kernel(float* w, const float* g, float* m, float* v, int64_t n, float lr,
                                                   float b1, float b2, float eps, float c1, float c2) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// Warm-start input: x[p] = (re, im) of u0[p] / scale (complex64 planar ->
// NHWC fp32, 2 channels), and per-block partial sums of |u0|^2.
// Scale of the warm-start network input: the RMS of A^*f from its sum of
// squares ss (n pixels), 1 for an all-zero image.
__device__ __forceinline__ double ws_scale(const double* ss, int64_t n) {
  return ss[0] > 0 ? sqrt(ss[0] / double(n)) : 1.0;
}
__global__ __launch_bounds__(256) void ws_pack(const float2* u0, int64_t n, const double* ss, float* x) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float inv_scale = float(1.0 / ws_scale(ss, n));
  const float2 z = u0[i];
  x[2 * i] = z.x * inv_scale;
  x[2 * i + 1] = z.y * inv_scale;
}
__global__ __launch_bounds__(256) void ws_unpack(const float* x, const float* y, int64_t n, const double* ss,
                                                 float2* u, float2* v) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float scale = float(ws_scale(ss, n));
  const float* yi = y + 6 * i;
  u[i] = make_float2(scale * (x[2 * i] + yi[0]), scale * (x[2 * i + 1] + yi[1]));
  v[i] = make_float2(scale * yi[2], scale * yi[3]);
  v[n + i] = make_float2(scale * yi[4], scale * yi[5]);
}

}  // namespace

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
bool cnn_layer_supported(int cin, int cout) {
  return (cin == 2 && cout == 32) || (cin == 32 && cout == 32) || (cin == 32 && cout == 6);
}

// A convolution whose kernel keeps `waves` waves per SIMD resident.
#define PDT_CONV(waves, kern, ...) \
  hipLaunchKernelGGL(kern, dim3(conv_blocks(n, h, w, waves)), dim3(kConvThreads), 0, st, __VA_ARGS__, n, h, w)
constexpr int kWaves32 = 2, kWavesLast = 3, kWavesIn = 8, kWaves8 = 6;

void cnn_conv_first(hipStream_t st, const float* x, const void* wk, const float* b, void* out, int n, int h, int w) {
  PDT_CONV(kWavesIn, conv_in_kernel, x, static_cast<const bf8*>(wk), b, static_cast<__bf16*>(out));
}
void cnn_conv_hidden(hipStream_t st, const void* in, const void* wk, const float* b, void* out, int n, int h, int w) {
  PDT_CONV(kWaves32, (conv32_kernel<2, EPI_RELU_BF16>), static_cast<const __bf16*>(in), static_cast<const bf8*>(wk), b, out,
           nullptr, nullptr);
}
void cnn_conv_last(hipStream_t st, const void* in, const void* wk, const float* b, float* y, int n, int h, int w) {
  PDT_CONV(kWavesLast, (conv32_kernel<1, EPI_F32>), static_cast<const __bf16*>(in), static_cast<const bf8*>(wk), b, y, nullptr,
           nullptr);
}
int cnn_net_rows(int depth, int n, int h, int w) {
  if (depth < 2 || depth > kNetLayers) return 0;
  const int ow = kNetCols - 2 * (depth - 1);
  const int64_t strips = int64_t(n) * ((w + ow - 1) / ow);
  const double kpx = 1e-3 * n * h * w;
  double best = 3.9 * depth + kpx * (0.031 + 0.034 * (depth - 2));
  const double step = depth == 2 ? 0.28 : depth <= 5 ? 0.45 : depth == 6 ? 0.50 : 0.69;
  int rows = 0;
  for (int rounds = 1; rounds <= 32; ++rounds) {
    const int64_t chunks = kNetBlocks * rounds / strips;
    if (chunks == 0) continue;
    const int R = int((h + chunks - 1) / chunks + 2) / 3 * 3;
    const double t = rounds * (1.4 + step * net_steps(R, depth));
    if (t < best) best = t, rows = R;
  }
  return rows;
}
void cnn_net(hipStream_t st, const CnnLayer* ls, int depth, const float* x, float* y, int n, int h, int w, int rows) {
  const int ow = kNetCols - 2 * (depth - 1), ns = (w + ow - 1) / ow;
  CnnLayers t{};
  for (int l = 0; l < depth; ++l) t.l[l] = ls[l];
  hipLaunchKernelGGL(net_kernel, dim3(n * ns * ((h + rows - 1) / rows)), dim3(64 * depth), 0, st, x, y, t, depth, n, h, w,
                     rows);
}

void cnn_conv_last_mse(hipStream_t st, const void* in, const void* wk, const float* b, const float* t, void* dz,
                       double* part, int n, int h, int w) {
  PDT_CONV(kWavesLast, (conv32_kernel<1, EPI_MSE>), static_cast<const __bf16*>(in), static_cast<const bf8*>(wk), b, dz, t, part);
}
int cnn_mse_blocks(int n, int h, int w) { return conv_blocks(n, h, w, kWavesLast); }

void cnn_conv_backward_data(hipStream_t st, int cout, const void* dz, const void* wt, const void* act, void* din, int n,
                            int h, int w) {
  const __bf16* z = static_cast<const __bf16*>(dz);
  const bf8* k = static_cast<const bf8*>(wt);
  if (cout == 32) PDT_CONV(kWaves32, (conv32_kernel<2, EPI_MASK_BF16>), z, k, nullptr, din, act, nullptr);
  else PDT_CONV(kWaves8, conv8_kernel, z, k, static_cast<__bf16*>(din), static_cast<const __bf16*>(act));
}

// Blocks of the weight-gradient kernels: at least 4 strip rows per wave.
static int wgrad_blocks(int n, int h, int w) {
  const int64_t rows = int64_t(n) * h * ((w + kGradStrip - 1) / kGradStrip);
  const int64_t b = (rows + 4 * kGradWaves - 1) / (4 * kGradWaves);
  return int(b < kGradBlocks ? b : kGradBlocks);
}
size_t cnn_wgrad_part_floats(int cin, int cout, int n, int h, int w) {
  return size_t(wgrad_blocks(n, h, w)) * grad_floats(cin, cout);
}

void cnn_conv_wgrad(hipStream_t st, CnnLayer& L, const void* in, const void* dz, int n, int h, int w) {
  const __bf16* z = static_cast<const __bf16*>(dz);
  const __bf16* x = static_cast<const __bf16*>(in);
  L.nblk = wgrad_blocks(n, h, w);
  const dim3 grid(L.nblk), block(kGradThreads);
  if (L.cin == 2) hipLaunchKernelGGL(wgrad_in_kernel, grid, block, 0, st, static_cast<const float*>(in), z, L.part, n, h, w);
  else if (L.cout == 32) hipLaunchKernelGGL((wgrad32_kernel<32>), grid, block, 0, st, x, z, L.part, n, h, w);
  else hipLaunchKernelGGL((wgrad32_kernel<6>), grid, block, 0, st, x, z, L.part, n, h, w);
}

// One launch over at most kCnnLayers layers at a time.
template <class F>
static void over_layers(const CnnLayer* ls, int count, F&& launch) {
  for (int i = 0; i < count; i += kCnnLayers) {
    CnnLayers t{};
    const int m = count - i < kCnnLayers ? count - i : kCnnLayers;
    for (int k = 0; k < m; ++k) t.l[k] = ls[i + k];
    launch(t, m);
  }
}

void cnn_reduce_grads(hipStream_t st, const CnnLayer* ls, int count) {
  over_layers(ls, count, [&](const CnnLayers& t, int m) {
    int most = 0;
    for (int k = 0; k < m; ++k) most = grad_floats(t.l[k].cin, t.l[k].cout) > most ? grad_floats(t.l[k].cin, t.l[k].cout) : most;
    hipLaunchKernelGGL(wgrad_reduce, dim3((most + kRedOut - 1) / kRedOut, m), dim3(kRedOut * kRedGroups), 0, st, t);
  });
}

size_t cnn_wk_elems(int cin, int cout) { return size_t(ksteps(cin)) * tiles_out(cout) * 512; }

void cnn_pack_weights(hipStream_t st, const CnnLayer* ls, int count) {
  over_layers(ls, count, [&](CnnLayers t, int m) {
    int most = 0;
    for (int k = 0; k < m; ++k) {
      CnnLayer& L = t.l[k];
      L.nk = int(cnn_wk_elems(L.cin, L.cout));
      L.nt = int(cnn_wk_elems(L.cout, L.cin));
      most = L.nk > most ? L.nk : most;
      most = L.nt > most ? L.nt : most;
    }
    hipLaunchKernelGGL(pack_weights, dim3((most + 255) / 256, m), dim3(256), 0, st, t);
  });
}

void cnn_adam(hipStream_t st, float* w, const float* g, float* m, float* v, int64_t n, float lr, float b1, float b2,
              float eps, float c1, float c2) {
  hipLaunchKernelGGL(adam_kernel, dim3(int((n + 255) / 256)), dim3(256), 0, st, w, g, m, v, n, lr, b1, b2, eps, c1, c2);
}

void cnn_ws_pack(hipStream_t st, const void* u0, int64_t n, const double* ss, float* x) {
  hipLaunchKernelGGL(ws_pack, dim3(int((n + 255) / 256)), dim3(256), 0, st, static_cast<const float2*>(u0), n, ss,
                     x);
}

void cnn_ws_unpack(hipStream_t st, const float* x, const float* y, int64_t n, const double* ss, void* u, void* v) {
  hipLaunchKernelGGL(ws_unpack, dim3(int((n + 255) / 256)), dim3(256), 0, st, x, y, n, ss,
                     static_cast<float2*>(u), static_cast<float2*>(v));
}

}  // namespace pdt
