// pdt_kernels.hip -- CDNA4 (gfx950) kernels of the TV/TGV primal-dual solvers.
//
// Design (one launch per half-iteration, batched over slices):
//  * Denoising (TvOptimizer / TgvOptimizer): each half-iteration is one
//    kernel over row-block work items that fuses the forward/backward
//    difference stencils, the dual ascent with its pointwise ball projection
//    and the over-relaxed primal step (tgv_kernels.cuh:225-324,568-605,647-686).
//  * Cartesian MRI (TgvMriOptimizer and the with-operator solvers): three
//    kernels per iteration.
//      rows_fwd  : dual p (and q) update of image row y, then for every coil
//                  S_c * u_bar row, ifftshift, PE-FFT in LDS, fftshift, keep
//                  the sampled PE columns                  -> T1 [c][y][ks]
//      cols      : per coil and group of sampled columns: FE-FFT of the
//                  zero-padded (read-out oversampled) column, mask, data prox
//                  of r, mask, inverse FE-FFT, crop to the image window
//                                                           -> T2 [c][y][ks]
//      rows_adj  : inverse PE-FFT of every coil's row, conj(S_c) coil sum
//                  (deterministic, in registers), then the primal u (and v)
//                  step of row y.
//    This replaces prefft/applyMask/preifft/combineImg/padFOV/cropFOV, the
//    cuFFT calls and TGV_prox_r/TGV_dual_*/TGV_primal_* of the reference
//    (mricartesianoperator.cu:28-160,196-414; tgvmrioptimizer.cu:162-198).
//  * The FFT is a mixed-radix Stockham autosort in LDS with radix-2/3/4/5/8
//    register codelets and a generic odd-prime stage (e.g. 23 for 368/736).
//  * Gap terms are accumulated in double per work item on evaluation
//    iterations only (template GAP), and reduced per slice in a fixed order.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <functional>
#include <mutex>
#include <type_traits>

#include "pdt_desc.hpp"
#include "pdt_launch.hpp"
#include "pdt_pixel.hpp"

namespace pdt {

// ---------------------------------------------------------------------------
// Block reductions (wave64 shuffles, then the 4 waves in a fixed order)
// ---------------------------------------------------------------------------
template <int N, int NT = kBlock>
__device__ __forceinline__ void block_sum(double (&v)[N], double* out) {
  __shared__ double red[(NT / 64) * kGapTerms];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int t = 0; t < N; ++t) {
    double x = v[t];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x += __shfl_down(x, o, 64);
    if (lane == 0) red[wave * kGapTerms + t] = x;
  }
  __syncthreads();
  if (threadIdx.x < N) {
    double s = 0;
    for (int w = 0; w < NT / 64; ++w) s += red[w * kGapTerms + threadIdx.x];
    out[threadIdx.x] = s;
  }
}

// block_sum for a block of blockDim.x threads (a multiple of 64, at most 1024).
template <int N>
__device__ __forceinline__ void block_sum_dyn(double (&v)[N], double* out) {
  __shared__ double red[16 * kGapTerms];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
  for (int t = 0; t < N; ++t) {
    double x = v[t];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x += __shfl_down(x, o, 64);
    if (lane == 0) red[wave * kGapTerms + t] = x;
  }
  __syncthreads();
  if (threadIdx.x < N) {
    double s = 0;
    for (int w = 0; w < nw; ++w) s += red[w * kGapTerms + threadIdx.x];
    out[threadIdx.x] = s;
  }
}

template <int NT = kBlock>
__device__ __forceinline__ double block_max(double v) {
  __shared__ double red[NT / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_down(v, o, 64));
  if (lane == 0) red[wave] = v;
  __syncthreads();
  double m = red[0];
  for (int w = 1; w < NT / 64; ++w) m = fmax(m, red[w]);
  return m;
}

// ---------------------------------------------------------------------------
// Mixed-radix Stockham FFT in LDS
//   stage radix r, p = product of earlier radices, nr = n / r:
//   for i in [0, nr): k = i mod p,
//     x_j = in[i + j nr] * w_n^(j k n/(p r)),  y = DFT_r(x),
//     out[(i - k) r + k + q p] = y_q.
// ---------------------------------------------------------------------------
template <class R>
__device__ __forceinline__ Cx<R> twd(const Cx<R>* tw, int m, bool inv) {
  Cx<R> w = tw[m];
  if (inv) w.im = -w.im;
  return w;
}
// x * (s i), s = +1 / -1
template <class R> __device__ __forceinline__ Cx<R> muli(Cx<R> x, R s) { return {-s * x.im, s * x.re}; }

template <class R, int RR> struct Dft;
template <class R> struct Dft<R, 2> {
  static __device__ __forceinline__ void run(Cx<R>* x, R) {
    Cx<R> a = x[0], b = x[1];
    x[0] = a + b;
    x[1] = a - b;
  }
};
template <class R> struct Dft<R, 3> {
  static __device__ __forceinline__ void run(Cx<R>* x, R s) {
    const R h = R(0.86602540378443864676);
    Cx<R> t = x[1] + x[2];
    Cx<R> d = muli(x[1] - x[2], s) * h;
    Cx<R> m = x[0] - t * R(0.5);
    x[0] = x[0] + t;
    x[1] = m + d;
    x[2] = m - d;
  }
};
template <class R> struct Dft<R, 4> {
  static __device__ __forceinline__ void run(Cx<R>* x, R s) {
    Cx<R> t0 = x[0] + x[2], t1 = x[0] - x[2], t2 = x[1] + x[3], t3 = muli(x[1] - x[3], s);
    x[0] = t0 + t2;
    x[2] = t0 - t2;
    x[1] = t1 + t3;
    x[3] = t1 - t3;
  }
};
template <class R> struct Dft<R, 5> {
  static __device__ __forceinline__ void run(Cx<R>* x, R s) {
    const R c1 = R(0.30901699437494742410), c2 = R(-0.80901699437494742410);
    const R s1 = R(0.95105651629515357212), s2 = R(0.58778525229247312917);
    Cx<R> t1 = x[1] + x[4], t2 = x[2] + x[3], d1 = x[1] - x[4], d2 = x[2] - x[3];
    Cx<R> a1 = x[0] + t1 * c1 + t2 * c2;
    Cx<R> a2 = x[0] + t1 * c2 + t2 * c1;
    Cx<R> b1 = muli(d1 * s1 + d2 * s2, s);
    Cx<R> b2 = muli(d1 * s2 - d2 * s1, s);
    x[0] = x[0] + t1 + t2;
    x[1] = a1 + b1;
    x[4] = a1 - b1;
    x[2] = a2 + b2;
    x[3] = a2 - b2;
  }
};
template <class R> struct Dft<R, 8> {
  static __device__ __forceinline__ void run(Cx<R>* x, R s) {
    Cx<R> e[4] = {x[0], x[2], x[4], x[6]};
    Cx<R> o[4] = {x[1], x[3], x[5], x[7]};
    Dft<R, 4>::run(e, s);
    Dft<R, 4>::run(o, s);
    const R c = R(0.70710678118654752440);
    Cx<R> w1 = {c, s * c}, w3 = {-c, s * c};
    Cx<R> o1 = o[1] * w1, o2 = muli(o[2], s), o3 = o[3] * w3;
    x[0] = e[0] + o[0];
    x[4] = e[0] - o[0];
    x[1] = e[1] + o1;
    x[5] = e[1] - o1;
    x[2] = e[2] + o2;
    x[6] = e[2] - o2;
    x[3] = e[3] + o3;
    x[7] = e[3] - o3;
  }
};

// Radices 6, 10 and 12.  6 and 10: even/odd split into two DFTs of half length m,
// X[k] = E[k] + w^k O[k], X[k + m] = E[k] - w^k O[k], w = exp(s i pi / m).
template <class R> struct Dft<R, 6> {
  static __device__ __forceinline__ void run(Cx<R>* x, R s) {
    Cx<R> e[3] = {x[0], x[2], x[4]};
    Cx<R> o[3] = {x[1], x[3], x[5]};
    Dft<R, 3>::run(e, s);
    Dft<R, 3>::run(o, s);
    const R h = R(0.86602540378443864676);  // sin(pi / 3)
    const Cx<R> t1 = o[1] * Cx<R>{R(0.5), s * h}, t2 = o[2] * Cx<R>{R(-0.5), s * h};
    x[0] = e[0] + o[0];
    x[3] = e[0] - o[0];
    x[1] = e[1] + t1;
    x[4] = e[1] - t1;
    x[2] = e[2] + t2;
    x[5] = e[2] - t2;
  }
};
template <class R> struct Dft<R, 12> {
  // X[k + 4 m] = sum_j w3^(j m) w12^(j k) Y_j[k], Y_j the 4-point DFT of
  // x[j], x[j + 3], x[j + 6], x[j + 9]
  static __device__ __forceinline__ void run(Cx<R>* x, R s) {
    const R h = R(0.86602540378443864676);  // cos(pi / 6)
    Cx<R> y[3][4];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
#pragma unroll
      for (int i = 0; i < 4; ++i) y[j][i] = x[j + 3 * i];
      Dft<R, 4>::run(y[j], s);
    }
    y[1][1] = y[1][1] * Cx<R>{h, s * R(0.5)};
    y[1][2] = y[1][2] * Cx<R>{R(0.5), s * h};
    y[1][3] = muli(y[1][3], s);
    y[2][1] = y[2][1] * Cx<R>{R(0.5), s * h};
    y[2][2] = y[2][2] * Cx<R>{R(-0.5), s * h};
    y[2][3] = -y[2][3];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      Cx<R> z[3] = {y[0][k], y[1][k], y[2][k]};
      Dft<R, 3>::run(z, s);
      x[k] = z[0];
      x[k + 4] = z[1];
      x[k + 8] = z[2];
    }
  }
};
template <class R> struct Dft<R, 10> {
  static __device__ __forceinline__ void run(Cx<R>* x, R s) {
    Cx<R> e[5] = {x[0], x[2], x[4], x[6], x[8]};
    Cx<R> o[5] = {x[1], x[3], x[5], x[7], x[9]};
    Dft<R, 5>::run(e, s);
    Dft<R, 5>::run(o, s);
    // cos and sin of k pi / 5, k = 1, 2
    const R c1 = R(0.80901699437494742410), c2 = R(0.30901699437494742410);
    const R s1 = R(0.58778525229247312917), s2 = R(0.95105651629515357212);
    Cx<R> t[5];
    t[0] = o[0];
    t[1] = o[1] * Cx<R>{c1, s * s1};
    t[2] = o[2] * Cx<R>{c2, s * s2};
    t[3] = o[3] * Cx<R>{-c2, s * s2};
    t[4] = o[4] * Cx<R>{-c1, s * s1};
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      x[k] = e[k] + t[k];
      x[k + 5] = e[k] - t[k];
    }
  }
};

template <class R, int RR>
__device__ __forceinline__ void butterfly(const Cx<R>* in, Cx<R>* out, int nr, int p,
                                          const Cx<R>* tw, int ts, bool inv) {
  Cx<R> x[RR];
  x[0] = in[0];
#pragma unroll
  for (int j = 1; j < RR; ++j) x[j] = in[j * nr] * twd(tw, j * ts, inv);
  Dft<R, RR>::run(x, inv ? R(1) : R(-1));
#pragma unroll
  for (int q = 0; q < RR; ++q) out[q * p] = x[q];
}

// One output q of a generic-radix butterfly (primes without a codelet):
// the stage twiddle w_n^(j ts) and the DFT factor w_r^(j q) = w_n^(j q nr) of
// input j are one table entry, w_n^(j step) with step = ts + q nr < n, its
// index stepped modulo n.
template <class R>
__device__ __forceinline__ Cx<R> dft_gen_output(const Cx<R>* in, int r, int nr, int step, int n, const Cx<R>* tw, R sg) {
  Cx<R> acc = in[0];
  int idx = step;
#pragma unroll 4
  for (int j = 1; j < r; ++j) {
    const Cx<R> x = in[j * nr], w = tw[idx];
    const R wi = sg * w.im;
    acc = {fma(-x.im, wi, fma(x.re, w.re, acc.re)), fma(x.im, w.re, fma(x.re, wi, acc.im))};
    idx += step;
    idx = idx >= n ? idx - n : idx;
  }
  return acc;
}

// cos and sin of 2 pi j / n at compile time (Taylor series on |x| <= pi / 2
// after the symmetries of the circle), for the odd-prime butterflies.
constexpr double ct_taylor_sin(double x) {
  double t = x, r = x;
  for (int k = 1; k < 14; ++k) {
    t *= -x * x / double((2 * k) * (2 * k + 1));
    r += t;
  }
  return r;
}
constexpr double ct_taylor_cos(double x) {
  double t = 1, r = 1;
  for (int k = 1; k < 14; ++k) {
    t *= -x * x / double((2 * k - 1) * (2 * k));
    r += t;
  }
  return r;
}
constexpr double ct_sincos2pi(int j, int n, bool want_sin) {
  j %= n;
  double sg = 1;
  if (2 * j > n) {  // angle in (pi, 2 pi): sin changes sign, cos does not
    j = n - j;
    if (want_sin) sg = -1;
  }
  constexpr double kPi = 3.14159265358979323846264338327950288;
  double x = 2 * kPi * double(j) / double(n);  // [0, pi]
  if (2 * x > kPi) {                          // (pi / 2, pi]: reflect about pi / 2
    x = kPi - x;
    return want_sin ? sg * ct_taylor_sin(x) : -ct_taylor_cos(x);
  }
  return want_sin ? sg * ct_taylor_sin(x) : ct_taylor_cos(x);
}
template <int P>
struct OddRoots {
  double c[P] = {}, s[P] = {};
  constexpr OddRoots() {
    for (int j = 0; j < P; ++j) {
      c[j] = ct_sincos2pi(j, P, false);
      s[j] = ct_sincos2pi(j, P, true);
    }
  }
};
template <int P>
constexpr OddRoots<P> kOddRoots{};

// Odd radix P (7, 11, 13, 23, ...) in the symmetric form: with
// s_m = x_m + x_(P-m), d_m = x_m - x_(P-m), m = 1..h, h = (P-1)/2,
//   X_0 = x_0 + sum_m s_m,
//   X_k, X_(P-k) = x_0 + sum_m cos(2 pi m k / P) s_m  +/-  i sg sum_m sin(2 pi m k / P) d_m,
// sg = -1 forward, +1 inverse: h^2 complex-by-real products per output pair.
// Both loops unroll, so the coefficients are compile-time constants rather
// than loads from the twiddle table.  in[j * nr] are the inputs, out[q * p]
// the outputs; tw (length-n table) supplies the stage twiddles only.  With
// G > 1 the call computes only the output pairs k = g + 1 (mod G) (and X_0
// for g = 0): G callers share one butterfly.
template <class R, int P>
__device__ __forceinline__ void butterfly_odd(const Cx<R>* in, Cx<R>* out, int nr, int p, const Cx<R>* tw,
                                              int ts, bool inv, int G = 1, int g = 0) {
  constexpr int h = (P - 1) / 2;
  const Cx<R> x0 = in[0];
  Cx<R> s[h], d[h];
  Cx<R> sum = x0;
#pragma unroll
  for (int m = 1; m <= h; ++m) {
    const Cx<R> a = in[m * nr] * twd(tw, m * ts, inv);
    const Cx<R> b = in[(P - m) * nr] * twd(tw, (P - m) * ts, inv);
    s[m - 1] = a + b;
    d[m - 1] = a - b;
    sum = sum + s[m - 1];
  }
  if (g == 0) out[0] = sum;
  const R sg = inv ? R(1) : R(-1);
#pragma unroll
  for (int k = 1; k <= h; ++k) {
    if (((k - 1) & (G - 1)) != g) continue;  // G is 1, 2 or 4
    Cx<R> A = x0, B = pzero<Cx<R>>();
#pragma unroll
    for (int m = 1; m <= h; ++m) {
      const int jk = (m * k) % P;
      A = A + s[m - 1] * R(kOddRoots<P>.c[jk]);
      B = B + d[m - 1] * R(kOddRoots<P>.s[jk]);
    }
    const Cx<R> iB = muli(B, sg);
    out[k * p] = A + iB;
    out[(P - k) * p] = A - iB;
  }
}

// Exact a / b for 0 <= a < 2^24, 1 <= b < 2^12 from a float reciprocal.
__device__ __forceinline__ int qdiv(int a, int b, float rb) {
  int q = __float2int_rz(float(a) * rb);
  if (q * b > a) --q;
  else if ((q + 1) * b <= a) ++q;
  return q;
}
// a / n where n == NF when NF > 0 (a division by a constant), else qdiv.
template <int NF>
__device__ __forceinline__ int divn(int a, int n, float rn) {
  if constexpr (NF > 0) return a / NF;
  else return qdiv(a, n, rn);
}


// Transforms nseq sequences of length pl.n stored back to back in a; b is
// scratch of the same size; tw is the twiddle table (LDS or global).
// Returns the buffer that holds the result.  Ends with a barrier.  Inlined,
// so that a and b stay LDS pointers (a call would pass generic ones and turn
// every access into a flat one) and the caller's registers need no saving.
template <class R, int NT>
__device__ __forceinline__ Cx<R>* lds_fft(Cx<R>* a, Cx<R>* b, int nseq, const FftPlanD& pl, const Cx<R>* tw, bool inv) {
  const int n = pl.n;
  for (int s = 0; s < pl.ns; ++s) {
    const int r = pl.r[s], nr = pl.nr[s], p = pl.p[s], tws = pl.tws[s];
    const float rnr = pl.rnr[s], rp = pl.rp[s];
    const bool p2 = (p & (p - 1)) == 0;  // uniform: power-of-two radices come first
    if (r == 2 || r == 3 || r == 4 || r == 5 || r == 8) {
      const int total = nseq * nr;
      for (int t = threadIdx.x; t < total; t += NT) {
        const int seq = nseq == 1 ? 0 : qdiv(t, nr, rnr);
        const int i = t - seq * nr;
        const int k = p2 ? (i & (p - 1)) : i - qdiv(i, p, rp) * p;
        const Cx<R>* in = a + seq * n + i;
        Cx<R>* out = b + seq * n + (i - k) * r + k;
        const int ts = k * tws;
        switch (r) {
          case 2: butterfly<R, 2>(in, out, nr, p, tw, ts, inv); break;
          case 3: butterfly<R, 3>(in, out, nr, p, tw, ts, inv); break;
          case 4: butterfly<R, 4>(in, out, nr, p, tw, ts, inv); break;
          case 5: butterfly<R, 5>(in, out, nr, p, tw, ts, inv); break;
          default: butterfly<R, 8>(in, out, nr, p, tw, ts, inv); break;
        }
      }
    } else {
      // Generic radix: a thread takes one output of a butterfly, not all r
      // of them.  A block holds few butterflies of a large prime (14 of
      // radix 31 in two columns of 217), so a thread per butterfly left
      // nearly every lane idle through r^2 products: 217 x 230, 8 coils,
      // 319 us per TGV iteration (k_cols alone 204 us), 43.5 us this way.
      const R sg = inv ? R(-1) : R(1);
      const int total = nseq * n;
      const float rn = 1.0f / float(n);
      for (int t = threadIdx.x; t < total; t += NT) {
        const int seq = nseq == 1 ? 0 : qdiv(t, n, rn);
        const int e = t - seq * n, q = qdiv(e, nr, rnr), i = e - q * nr;
        const int k = p2 ? (i & (p - 1)) : i - qdiv(i, p, rp) * p;
        b[seq * n + (i - k) * r + k + q * p] = dft_gen_output<R>(a + seq * n + i, r, nr, k * tws + q * nr, n, tw, sg);
      }
    }
    __syncthreads();
    Cx<R>* t = a;
    a = b;
    b = t;
  }
  return a;
}

// ---------------------------------------------------------------------------
// Compile-time-planned Stockham FFT for the common transform lengths.  The
// stage formula of lds_fft, with radix, stride and twiddle steps
// constant-folded; lengths without a specialisation use lds_fft.
// ---------------------------------------------------------------------------
constexpr int ct_radix(int n, int s) {
  // 384 and 640: a last stage of radix 6 or 10 instead of a radix-2 stage
  // followed by a radix-3 or radix-5 one (the first stage stays radix 8,
  // as the padded LDS layout requires).
  if (n == 384) return s < 2 ? 8 : s == 2 ? 6 : 1;
  if (n == 640) return s < 2 ? 8 : s == 2 ? 10 : 1;
  int k = 0;
  while (n % 8 == 0 && n > 8) {
    if (k == s) return 8;
    n /= 8;
    ++k;
  }
  const int small[5] = {8, 4, 2, 3, 5};
  for (int j = 0; j < 5; ++j)
    while (n % small[j] == 0 && n >= small[j]) {
      if (k == s) return small[j];
      n /= small[j];
      ++k;
    }
  for (int p = 7; n > 1; p += 2)
    while (n % p == 0) {
      if (k == s) return p;
      n /= p;
      ++k;
    }
  return 1;
}
constexpr int ct_nstages(int n) {
  int s = 0;
  while (ct_radix(n, s) != 1) ++s;
  return s;
}
// The padded LDS layout (element e at e + e / 8) keeps every input and
// output of a butterfly at a constant padded stride when n, every n / r and
// every earlier-radix product p (or r, when p = 1) are multiples of 8.
constexpr bool ct_pad_ok(int n) {
  if (n % 8 != 0) return false;
  int p = 1;
  for (int s = 0; s < ct_nstages(n); ++s) {
    const int r = ct_radix(n, s);
    if ((n / r) % 8 != 0 || (p == 1 ? r != 8 : p % 8 != 0)) return false;
    p *= r;
  }
  return true;
}

// Unpadded FFT buffers (the wide adjoint row pass, whose two buffers fill
// the LDS share of a workgroup) permute their slots instead: bits 0-2 of an
// element index are XORed with bits 4-6 and bit 3 with bit 6, a permutation
// of every aligned block of 16 elements.  The Stockham writes at strides of 8
// and 64 elements then spread the lanes of a wave over distinct banks, while
// runs of 16 consecutive elements (the reads) stay on distinct banks.
__device__ __forceinline__ int swz(int e) { return e ^ ((e >> 4) & 7) ^ (((e >> 6) & 1) << 3); }

// LDS slot of element e of an FFT buffer.  Kernels with a compile-time length
// (NF > 0) pad one element after every 8: the Stockham stages write with
// strides of 8 elements (and multiples), which would otherwise put the 64
// lanes of a wave on a few LDS banks.  Without padding (LP = false) the
// slots are permuted by swz.
template <int NF, bool LP = true>
__device__ __forceinline__ int lp(int e) {
  if constexpr (NF > 0 && ct_pad_ok(NF)) return LP ? e + (e >> 3) : swz(e);
  else return e;
}

// TW: stage twiddles present (false for the first stage, where they are 1).
// nr, p: LDS strides of the inputs and outputs.
template <class R, int RR, bool TW>
__device__ __forceinline__ void butterfly_ct(const Cx<R>* in, Cx<R>* out, int ts, const Cx<R>* tw, bool inv,
                                             int nr, int p) {
  if constexpr (RR == 2 || RR == 3 || RR == 4 || RR == 5 || RR == 6 || RR == 8 || RR == 10) {
    Cx<R> x[RR];
    x[0] = in[0];
#pragma unroll
    for (int j = 1; j < RR; ++j) x[j] = TW ? in[j * nr] * twd(tw, j * ts, inv) : in[j * nr];
    Dft<R, RR>::run(x, inv ? R(1) : R(-1));
#pragma unroll
    for (int q = 0; q < RR; ++q) out[q * p] = x[q];
  } else {
    static_assert(RR % 2 == 1, "even radices are 2, 4, 6, 8 and 10");
    butterfly_odd<R, RR>(in, out, nr, p, tw, ts, inv);
  }
}

// butterfly_ct on swz-permuted buffers: inputs at logical elements
// ein + j nr of a, outputs at eout + q p of b.
template <class R, int RR, bool TW>
__device__ __forceinline__ void butterfly_ct_swz(const Cx<R>* a, Cx<R>* b, int ein, int eout, int ts,
                                                 const Cx<R>* tw, bool inv, int nr, int p) {
  static_assert(RR == 2 || RR == 3 || RR == 4 || RR == 5 || RR == 6 || RR == 8 || RR == 10, "radix");
  Cx<R> x[RR];
  x[0] = a[swz(ein)];
#pragma unroll
  for (int j = 1; j < RR; ++j) x[j] = TW ? a[swz(ein + j * nr)] * twd(tw, j * ts, inv) : a[swz(ein + j * nr)];
  Dft<R, RR>::run(x, inv ? R(1) : R(-1));
#pragma unroll
  for (int q = 0; q < RR; ++q) b[swz(eout + q * p)] = x[q];
}

template <class R, int N, int S, int P, int NT, bool INV, bool LP>
__device__ __forceinline__ Cx<R>* fft_ct_stage(Cx<R>* a, Cx<R>* b, int nseq, const Cx<R>* tw) {
  if constexpr (S == ct_nstages(N)) {
    return a;
  } else {
    constexpr int r = ct_radix(N, S), nr = N / r, tws = N / (P * r);
    // padded layout (ct_pad_ok): every input and output of a butterfly
    // sits at a constant padded stride from its first one
    constexpr bool PAD = LP && ct_pad_ok(N);
    constexpr int NP = PAD ? N + N / 8 : N, nrp = PAD ? nr + nr / 8 : nr, pp = PAD && P > 1 ? P + P / 8 : P;
    const int total = nseq * nr;
    if constexpr (r > 8 && r % 2 == 1) {
      // Odd prime radix: a long chain of products per butterfly and few
      // butterflies per block, so the output pairs of each butterfly are
      // split over G waves (G = 4, 2 or 1, as many as keep every butterfly
      // in one pass).  Lane l of a wave takes butterfly 64 c + l and the
      // wave-uniform part g, so every part keeps constant coefficients.
      constexpr int NW = NT / 64;
      const int chunks = (total + 63) / 64;
      const int G = chunks * 4 <= NW ? 4 : chunks * 2 <= NW ? 2 : 1;
      const int lane = threadIdx.x & 63;
      const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // a scalar, so the parts branch per wave
      for (int q = wave; q < chunks * G; q += NW) {
        const int c = q / G, g = q - c * G;
        const int t = c * 64 + lane;
        if (t < total) {
          const int seq = t / nr;
          const int i = t - seq * nr;
          const int k = i % P;
          const int o = (i - k) * r + k;
          const int ip = PAD ? i + (i >> 3) : i, op = PAD ? o + (o >> 3) : o;
          butterfly_odd<R, r>(a + seq * NP + ip, b + seq * NP + op, nrp, pp, tw, k * tws, INV, G, g);
        }
      }
    } else {
      for (int t = threadIdx.x; t < total; t += NT) {
        const int seq = t / nr;
        const int i = t - seq * nr;
        const int k = i % P;
        const int o = (i - k) * r + k;
        if constexpr (!LP && ct_pad_ok(N)) {
          butterfly_ct_swz<R, r, (P > 1)>(a, b, seq * N + i, seq * N + o, k * tws, tw, INV, nr, P);
        } else {
          const int ip = PAD ? i + (i >> 3) : i, op = PAD ? o + (o >> 3) : o;
          butterfly_ct<R, r, (P > 1)>(a + seq * NP + ip, b + seq * NP + op, k * tws, tw, INV, nrp, pp);
        }
      }
    }
    __syncthreads();
    return fft_ct_stage<R, N, S + 1, P * r, NT, INV, LP>(b, a, nseq, tw);
  }
}

// FFT of length NF with a compile-time plan, or of length pl.n with the
// runtime plan when NF == 0.  Each FFT kernel is instantiated per length, so
// its register budget is that of its own plan only (the runtime plan with
// its radix switch needs several times the registers of a fixed one).
template <class R, int NT, bool INV, int NF, bool LP = true>
__device__ __forceinline__ Cx<R>* fft_n(Cx<R>* a, Cx<R>* b, int nseq, const FftPlanD& pl, const Cx<R>* tw) {
  if constexpr (NF > 0) return fft_ct_stage<R, NF, 0, 1, NT, INV, LP>(a, b, nseq, tw);
  else return lds_fft<R, NT>(a, b, nseq, pl, tw, INV);
}

// One sequence of the compile-time plan transformed by one wavefront alone,
// in place on its padded slots (lengths with ct_pad_ok, at most 64 M
// butterflies per stage): each stage reads every input of the wave's
// butterflies into registers before it writes an output, and a wave's LDS
// accesses take effect in issue order, so no workgroup barrier separates the
// stages.  The butterflies are fft_ct_stage's (butterfly_ct's operations),
// so the result is that of fft_n on padded buffers.  seq: the sequence's
// first slot; call with S = 0, P = 1.
template <class R, int N, int S, int P, bool INV>
__device__ __forceinline__ void fft_wave(Cx<R>* seq, const Cx<R>* tw) {
  if constexpr (S < ct_nstages(N)) {
    constexpr int r = ct_radix(N, S), nr = N / r, tws = N / (P * r);
    static_assert(ct_pad_ok(N) && r <= 10, "wave transforms: padded lengths, register codelets");
    constexpr int nrp = nr + nr / 8, pp = P > 1 ? P + P / 8 : P;
    constexpr int M = (nr + 63) / 64;  // butterflies per lane
    const int lane = threadIdx.x & 63;
    Cx<R> x[M][r];
    int ob[M];
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const int i = lane + 64 * m;
      ob[m] = -1;
      if (i < nr) {
        const int k = i % P;
        const int o = (i - k) * r + k;
        const Cx<R>* in = seq + i + (i >> 3);
        x[m][0] = in[0];
#pragma unroll
        for (int j = 1; j < r; ++j) x[m][j] = P > 1 ? in[j * nrp] * twd(tw, j * (k * tws), INV) : in[j * nrp];
        Dft<R, r>::run(x[m], INV ? R(1) : R(-1));
        ob[m] = o + (o >> 3);
      }
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int m = 0; m < M; ++m)
      if (ob[m] >= 0) {
#pragma unroll
        for (int q = 0; q < r; ++q) seq[ob[m] + q * pp] = x[m][q];
      }
    __builtin_amdgcn_wave_barrier();
    fft_wave<R, N, S + 1, P * r, INV>(seq, tw);
  }
}

// numpy shift maps: ifftshift moves i to (i + ceil(n/2)) % n (the prefft /
// preifft index map of mricartesianoperator.cu:44-49); fftshift output k
// reads input (k - n/2) mod n.
// Both take 0 <= i < n and avoid the integer modulo.
__device__ __forceinline__ int ishift_dst(int i, int n) {
  const int j = i + (n + 1) / 2;
  return j >= n ? j - n : j;
}
__device__ __forceinline__ int fshift_src(int k, int n) {
  const int j = k + n - n / 2;
  return j >= n ? j - n : j;
}
// ifftshift gather: position j of ifftshift(z) holds z[(j + n/2) mod n].
__device__ __forceinline__ int ishift_src(int j, int n) {
  const int i = j + n / 2;
  return i >= n ? i - n : i;
}

// ---------------------------------------------------------------------------
// Stencil helpers on plane pointers (tgv_kernels.cuh:25-135)
// ---------------------------------------------------------------------------
// Both neighbours are loaded unconditionally (the first row / column reads
// its own element twice) and the boundary cases selected afterwards, so the
// loads issue together instead of behind branches.
template <class P, class S>
__device__ __forceinline__ P dmx(const S* a, int x, size_t i, int W) {
  using L = Ld<P, Plain<S>>;
  const P c = L::get(a, i), m = L::get(a, x > 0 ? i - 1 : i);
  const P d = (x < W - 1) ? c - m : -m;
  return x > 0 ? d : c;
}
template <class P, class S>
__device__ __forceinline__ P dmy(const S* a, int y, size_t i, int W, int H) {
  using L = Ld<P, Plain<S>>;
  const P c = L::get(a, i), m = L::get(a, y > 0 ? i - W : i);
  const P d = (y < H - 1) ? c - m : -m;
  return y > 0 ? d : c;
}

template <class R>
__device__ __forceinline__ R sched_alpha(const SliceDev& d, double a_start, double a_end, int k) {
  if (!d.schedule) return R(a_start);
  // tgvmrioptimizer.cu:150-155, evaluated in the solver's precision
  const R dk = R(k), dmax = R(d.kmax);
  return exp(dk / dmax * log(R(a_end)) + (dmax - dk) / dmax * log(R(a_start)));
}

// Dual ascent + projection of p (and q) at one pixel (dual_math on the
// pixel's values in memory).
template <class P, class S, bool TGV, bool GAP>
__device__ __forceinline__ void dual_pixel(const SliceDev& d, int x, int y, typename RealOf<P>::T sigma,
                                           Ball<typename RealOf<P>::T> w0, Ball<typename RealOf<P>::T> w1,
                                           double* t) {
  using L = Ld<P, S>;
  const int W = d.W, H = d.H;
  const size_t n = size_t(W) * H;
  const size_t i = size_t(y) * W + x;
  const size_t ixp = i + (x < W - 1), iyp = i + ((y < H - 1) ? W : 0);
  const auto ub = gptr<const P>(d.ub);
  const auto px = gptr<S>(d.p);
  const auto py = px + n;
  P vx0 = pzero<P>(), vy0 = vx0, vxx = vx0, vyx = vx0, vxy = vx0, vyy = vx0;
  P qxx = vx0, qyy = vx0, qxy = vx0;
  const auto qxxp = gptr<S>(d.q);
  const auto qyyp = qxxp + n;
  const auto qxyp = qyyp + n;
  if (TGV) {
    const auto vbx = gptr<const P>(d.vb);
    const auto vby = vbx + n;
    vx0 = vbx[i];
    vy0 = vby[i];
    vxx = vbx[ixp];
    vyx = vby[ixp];
    vxy = vbx[iyp];
    vyy = vby[iyp];
    qxx = L::get(qxxp, i);
    qyy = L::get(qyyp, i);
    qxy = L::get(qxyp, i);
  }
  P pxv = L::get(px, i), pyv = L::get(py, i);
  dual_math<P, TGV, GAP>(ub[i], ub[ixp], ub[iyp], vx0, vy0, vxx, vyx, vxy, vyy, pxv, pyv, qxx, qyy, qxy, sigma, w0,
                         w1, t);
  if (TGV) {
    L::put(qxxp, i, qxx);
    L::put(qyyp, i, qyy);
    L::put(qxyp, i, qxy);
  }
  L::put(px, i, pxv);
  L::put(py, i, pyv);
}

// v-step of TGV_primal_v_kernel (tgv_kernels.cuh:647-686) at one pixel;
// returns |p + div_sym q|^2 for the gap.
template <class P, class S>
__device__ __forceinline__ double vstep_pixel(const SliceDev& d, int x, int y, typename RealOf<P>::T tau,
                                              typename RealOf<P>::T theta) {
  using R = typename RealOf<P>::T;
  using L = Ld<P, S>;
  const int W = d.W, H = d.H;
  const size_t n = size_t(W) * H;
  const size_t i = size_t(y) * W + x;
  const auto px = gptr<const S>(d.p);
  const auto py = px + n;
  const auto qxx = gptr<const S>(d.q);
  const auto qyy = qxx + n;
  const auto qxy = qyy + n;
  const auto vx = gptr<P>(d.v);
  const auto vy = vx + n;
  const auto vbx = gptr<P>(d.vb);
  const auto vby = vbx + n;
  const P dsx = dmx<P>(qxx, x, i, W) + dmy<P>(qxy, y, i, W, H);
  const P dsy = dmy<P>(qyy, y, i, W, H) + dmx<P>(qxy, x, i, W);
  const P pxi = L::get(px, i), pyi = L::get(py, i);
  const P ox = vx[i], oy = vy[i];
  const P nx = ox + tau * (dsx + pxi);
  const P ny = oy + tau * (dsy + pyi);
  vx[i] = nx;
  vy[i] = ny;
  vbx[i] = (R(1) + theta) * nx - theta * ox;
  vby[i] = (R(1) + theta) * ny - theta * oy;
  return dabs2(pxi + dsx) + dabs2(pyi + dsy);
}

// ---------------------------------------------------------------------------
// Denoising half-iterations.  Item = (slice, first row); rpi rows per item.
// ---------------------------------------------------------------------------

// TV_dual_p_kernel (tgv_kernels.cuh:294-324).  Gap: P(ubar) terms.
template <class P, bool GAP, int NT>
__global__ __launch_bounds__(NT) void k_tv_dual(const SliceDev* sl, const int2* items, int rpi,
                                                    double* part) {
  const int bi = xcd_item(blockIdx.x, gridDim.x);  // neighbouring rows on one XCD
  const int2 it = items ? items[bi] : make_int2(0, bi * rpi);
  const SliceDev& d = sl[it.x];
  if (!slice_active(d)) return;
  using R = typename RealOf<P>::T;
  const int W = d.W, H = d.H;
  const int ya = it.y, yb = min(H, ya + rpi);
  const R sigma = R(d.sigma);
  const auto ub = gptr<const P>(d.ub);
  const auto f = gptr<const P>(d.f);
  double t[kGapTerms] = {0};
  const int cnt = (yb - ya) * W;
  for (int idx = threadIdx.x; idx < cnt; idx += NT) {
    const int yy = idx / W;
    const int x = idx - yy * W, y = ya + yy;
    dual_pixel<P, P, false, GAP>(d, x, y, sigma, ball_any(R(1)), ball_any(R(1)), t);
    if (GAP) {
      const size_t i = size_t(y) * W + x;
      t[3] += dabs2(ub[i] - f[i]);
    }
  }
  if (GAP) block_sum<4, NT>(reinterpret_cast<double(&)[4]>(t), part + size_t(bi) * kGapTerms);
}

// TV_primal_u_kernel 2D (tgv_kernels.cuh:568-605).  Gap: ROF dual terms
// Re<div p, f>, ||div p||^2.
template <class P, bool GAP, int NT>
__global__ __launch_bounds__(NT) void k_tv_primal(const SliceDev* sl, const int2* items, int rpi,
                                                      double* part) {
  const int bi = xcd_item(blockIdx.x, gridDim.x);  // neighbouring rows on one XCD
  const int2 it = items ? items[bi] : make_int2(0, bi * rpi);
  const SliceDev& d = sl[it.x];
  if (!slice_active(d)) return;
  using R = typename RealOf<P>::T;
  const int W = d.W, H = d.H;
  const size_t n = size_t(W) * H;
  const int ya = it.y, yb = min(H, ya + rpi);
  const R tau = R(d.tau), lambda = R(d.lambda), theta = R(d.theta);
  const auto u = gptr<P>(d.u);
  const auto ub = gptr<P>(d.ub);
  const auto f = gptr<const P>(d.f);
  const auto px = gptr<const P>(d.p);
  const auto py = px + n;
  double t[2] = {0, 0};
  const int cnt = (yb - ya) * W;
  for (int idx = threadIdx.x; idx < cnt; idx += NT) {
    const int yy = idx / W;
    const int x = idx - yy * W, y = ya + yy;
    const size_t i = size_t(y) * W + x;
    const P uo = u[i];
    const P div = dmx<P>(px, x, i, W) + dmy<P>(py, y, i, W, H);
    P un = uo + tau * fmadd(lambda, P(f[i]), div);
    un = un * rcp(R(1) + tau * lambda);
    u[i] = un;
    ub[i] = (R(1) + theta) * un - theta * uo;
    if (GAP) {
      t[0] += redot(div, f[i]);
      t[1] += dabs2(div);
    }
  }
  if (GAP) block_sum<2, NT>(t, part + size_t(bi) * kGapTerms);
  if (ya == 0 && threadIdx.x == 0) gptr<int>(d.ctl)[CTL_ITER] += 1;
}

// TGV denoising primal half (tgvoptimizer.cu:119-127): TV_primal_u_kernel
// then TGV_primal_v_kernel at every pixel.
template <class P, class S, int NT>
__global__ __launch_bounds__(NT) void k_tgv_primal(const SliceDev* sl, const int2* items, int rpi) {
  const int bi = xcd_item(blockIdx.x, gridDim.x);  // neighbouring rows on one XCD
  const int2 it = items ? items[bi] : make_int2(0, bi * rpi);
  const SliceDev& d = sl[it.x];
  if (!slice_active(d)) return;
  using R = typename RealOf<P>::T;
  const int W = d.W, H = d.H;
  const size_t n = size_t(W) * H;
  const int ya = it.y, yb = min(H, ya + rpi);
  const R tau = R(d.tau), lambda = R(d.lambda), theta = R(d.theta);
  const auto u = gptr<P>(d.u);
  const auto ub = gptr<P>(d.ub);
  const auto f = gptr<const P>(d.f);
  const auto px = gptr<const S>(d.p);
  const auto py = px + n;
  const int cnt = (yb - ya) * W;
  for (int idx = threadIdx.x; idx < cnt; idx += NT) {
    const int yy = idx / W;
    const int x = idx - yy * W, y = ya + yy;
    const size_t i = size_t(y) * W + x;
    const P uo = u[i];
    const P div = dmx<P>(px, x, i, W) + dmy<P>(py, y, i, W, H);
    P un = uo + tau * fmadd(lambda, P(f[i]), div);
    un = un * rcp(R(1) + tau * lambda);
    u[i] = un;
    ub[i] = (R(1) + theta) * un - theta * uo;
    vstep_pixel<P, S>(d, x, y, tau, theta);
  }
}

// TGV denoising dual half (tgvoptimizer.cu:130-136).  Gap: P(ubar, vbar).
template <class P, class S, bool GAP, int NT>
__global__ __launch_bounds__(NT) void k_tgv_dual(const SliceDev* sl, const int2* items, int rpi,
                                                     double* part) {
  const int bi = xcd_item(blockIdx.x, gridDim.x);  // neighbouring rows on one XCD
  const int2 it = items ? items[bi] : make_int2(0, bi * rpi);
  const SliceDev& d = sl[it.x];
  if (!slice_active(d)) return;
  using R = typename RealOf<P>::T;
  const int W = d.W, H = d.H;
  const int ya = it.y, yb = min(H, ya + rpi);
  const R sigma = R(d.sigma);
  const auto w0 = ball_any(R(d.alpha0)), w1 = ball_any(R(d.alpha1));
  const auto ub = gptr<const P>(d.ub);
  const auto f = gptr<const P>(d.f);
  double t[kGapTerms] = {0};
  const int cnt = (yb - ya) * W;
  for (int idx = threadIdx.x; idx < cnt; idx += NT) {
    const int yy = idx / W;
    const int x = idx - yy * W, y = ya + yy;
    dual_pixel<P, S, true, GAP>(d, x, y, sigma, w0, w1, t);
    if (GAP) {
      const size_t i = size_t(y) * W + x;
      t[3] += dabs2(ub[i] - f[i]);
    }
  }
  if (GAP) block_sum<4, NT>(reinterpret_cast<double(&)[4]>(t), part + size_t(bi) * kGapTerms);
  if (ya == 0 && threadIdx.x == 0) gptr<int>(d.ctl)[CTL_ITER] += 1;
}

// Two pixels of storage type S side by side (one 8- or 16-byte access).
template <class S> struct alignas(2 * sizeof(S)) Pair {
  S a, b;
};

// k_tgv_dual with two horizontally adjacent pixels per thread (W even): the
// duals, ubar and vbar move as 2-pixel vectors (8 bytes per p, q plane access
// with fp16 storage, 16 with float2), the arithmetic is dual_math per pixel,
// so the iterates equal k_tgv_dual's bit for bit.
template <class P, class S, bool GAP, int NT>
__global__ __launch_bounds__(NT) void k_tgv_dual2(const SliceDev* sl, const int2* items, int rpi, double* part) {
  const int bi = xcd_item(blockIdx.x, gridDim.x);  // neighbouring rows on one XCD
  const int2 it = items ? items[bi] : make_int2(0, bi * rpi);
  const SliceDev& d = sl[it.x];
  if (!slice_active(d)) return;
  using R = typename RealOf<P>::T;
  using L = Ld<P, S>;
  const int W = d.W, H = d.H;
  const size_t n = size_t(W) * H;
  const int ya = it.y, yb = min(H, ya + rpi);
  const R sigma = R(d.sigma);
  const auto w0 = ball_any(R(d.alpha0)), w1 = ball_any(R(d.alpha1));
  const auto ub = gptr<const P>(d.ub);
  const auto ubp = gptr<const Pair<P>>(d.ub);
  const auto vbx = gptr<const P>(d.vb);
  const auto vbxp = gptr<const Pair<P>>(d.vb);
  const auto f = gptr<const P>(d.f);
  const auto pp = gptr<Pair<S>>(d.p);
  const auto qp = gptr<Pair<S>>(d.q);
  const size_t n2 = n / 2;  // pairs per plane
  double t[kGapTerms] = {0};
  const int W2 = W / 2, cnt = (yb - ya) * W2;
  for (int idx = threadIdx.x; idx < cnt; idx += NT) {
    const int yy = idx / W2;
    const int x = 2 * (idx - yy * W2), y = ya + yy;
    const size_t i = size_t(y) * W + x, i2 = i / 2;
    const bool last = x + 2 >= W, bottom = y >= H - 1;
    const size_t dn2 = bottom ? i2 : i2 + W2;  // pair below (the pair itself on the last row)
    const Pair<P> u0 = ubp[i2], ud = ubp[dn2];
    const P u2 = last ? u0.b : ub[i + 2];
    const Pair<P> vx = vbxp[i2], vy = vbxp[n2 + i2], vxd = vbxp[dn2], vyd = vbxp[n2 + dn2];
    const P vx2 = last ? vx.b : vbx[i + 2], vy2 = last ? vy.b : vbx[n + i + 2];
    Pair<S> ps[2] = {pp[i2], pp[n2 + i2]};
    Pair<S> qs[3] = {qp[i2], qp[n2 + i2], qp[2 * n2 + i2]};
    P pxa = L::get(&ps[0].a, 0), pya = L::get(&ps[1].a, 0);
    P qxxa = L::get(&qs[0].a, 0), qyya = L::get(&qs[1].a, 0), qxya = L::get(&qs[2].a, 0);
    P pxb = L::get(&ps[0].b, 0), pyb = L::get(&ps[1].b, 0);
    P qxxb = L::get(&qs[0].b, 0), qyyb = L::get(&qs[1].b, 0), qxyb = L::get(&qs[2].b, 0);
    // pixel x (never the last column), then x + 1
    dual_math<P, true, GAP>(u0.a, u0.b, bottom ? u0.a : ud.a, vx.a, vy.a, vx.b, vy.b, bottom ? vx.a : vxd.a,
                            bottom ? vy.a : vyd.a, pxa, pya, qxxa, qyya, qxya, sigma, w0, w1, t);
    dual_math<P, true, GAP>(u0.b, last ? u0.b : u2, bottom ? u0.b : ud.b, vx.b, vy.b, last ? vx.b : vx2,
                            last ? vy.b : vy2, bottom ? vx.b : vxd.b, bottom ? vy.b : vyd.b, pxb, pyb, qxxb, qyyb,
                            qxyb, sigma, w0, w1, t);
    L::put(&ps[0].a, 0, pxa);
    L::put(&ps[0].b, 0, pxb);
    L::put(&ps[1].a, 0, pya);
    L::put(&ps[1].b, 0, pyb);
    L::put(&qs[0].a, 0, qxxa);
    L::put(&qs[0].b, 0, qxxb);
    L::put(&qs[1].a, 0, qyya);
    L::put(&qs[1].b, 0, qyyb);
    L::put(&qs[2].a, 0, qxya);
    L::put(&qs[2].b, 0, qxyb);
    pp[i2] = ps[0];
    pp[n2 + i2] = ps[1];
    qp[i2] = qs[0];
    qp[n2 + i2] = qs[1];
    qp[2 * n2 + i2] = qs[2];
    if (GAP) {
      t[3] += dabs2(u0.a - f[i]);
      t[3] += dabs2(u0.b - f[i + 1]);
    }
  }
  if (GAP) block_sum<4, NT>(reinterpret_cast<double(&)[4]>(t), part + size_t(bi) * kGapTerms);
  if (ya == 0 && threadIdx.x == 0) gptr<int>(d.ctl)[CTL_ITER] += 1;
}

// TGV dual restoration, step 1: d = div_sym q into tmp, per-item max |d|.
template <class P, class S>
__global__ __launch_bounds__(kBlock) void k_tgv_restore1(const SliceDev* sl, const int2* items, int rpi,
                                                         double* part) {
  const int bi = xcd_item(blockIdx.x, gridDim.x);  // neighbouring rows on one XCD
  const int2 it = items ? items[bi] : make_int2(0, bi * rpi);
  const SliceDev& d = sl[it.x];
  if (!slice_active(d)) return;
  const int W = d.W, H = d.H;
  const size_t n = size_t(W) * H;
  const int ya = it.y, yb = min(H, ya + rpi);
  const auto qxx = gptr<const S>(d.q);
  const auto qyy = qxx + n;
  const auto qxy = qyy + n;
  const auto dx = gptr<P>(d.tmp);
  const auto dy = dx + n;
  double m = 0;
  const int cnt = (yb - ya) * W;
  for (int idx = threadIdx.x; idx < cnt; idx += kBlock) {
    const int yy = idx / W;
    const int x = idx - yy * W, y = ya + yy;
    const size_t i = size_t(y) * W + x;
    const P a = dmx<P>(qxx, x, i, W) + dmy<P>(qxy, y, i, W, H);
    const P b = dmy<P>(qyy, y, i, W, H) + dmx<P>(qxy, x, i, W);
    dx[i] = a;
    dy[i] = b;
    m = fmax(m, sqrt(dabs2(a) + dabs2(b)));
  }
  m = block_max(m);
  if (threadIdx.x == 0) part[size_t(bi) * kGapTerms + 0] = m;
}

// Step 2: g = div d, Re<g, f>, ||g||^2.
template <class P>
__global__ __launch_bounds__(kBlock) void k_tgv_restore2(const SliceDev* sl, const int2* items, int rpi,
                                                         double* part) {
  const int bi = xcd_item(blockIdx.x, gridDim.x);  // neighbouring rows on one XCD
  const int2 it = items ? items[bi] : make_int2(0, bi * rpi);
  const SliceDev& d = sl[it.x];
  if (!slice_active(d)) return;
  const int W = d.W, H = d.H;
  const size_t n = size_t(W) * H;
  const int ya = it.y, yb = min(H, ya + rpi);
  const auto dx = gptr<const P>(d.tmp);
  const auto dy = dx + n;
  const auto f = gptr<const P>(d.f);
  double t[2] = {0, 0};
  const int cnt = (yb - ya) * W;
  for (int idx = threadIdx.x; idx < cnt; idx += kBlock) {
    const int yy = idx / W;
    const int x = idx - yy * W, y = ya + yy;
    const size_t i = size_t(y) * W + x;
    const P g = dmx<P>(dx, x, i, W) + dmy<P>(dy, y, i, W, H);
    t[0] += redot(g, f[i]);
    t[1] += dabs2(g);
  }
  block_sum<2>(t, part + size_t(bi) * kGapTerms);
}

// ---------------------------------------------------------------------------
// Cartesian MRI passes.  MODE: 0 operator only, 1 TV-with-op, 2 TGV
// (TGV-MRI and TGV-with-op).  Row items are (slice, image row).
// ---------------------------------------------------------------------------
enum { M_OP = 0, M_TV = 1, M_TGV = 2 };


// LDS layout of the row FFT passes: twiddles (W), two FFT buffers (cb * W
// each), listed columns (nc ints).
template <class C>
struct RowLds {
  C* tw;
  C* a;
  C* b;
  int* cols;
  __device__ RowLds(char* raw, int W, int cb, bool padded = true) {
    const int n = padded ? lds_pad(cb * W) : cb * W;
    tw = reinterpret_cast<C*>(raw);
    a = tw + W;
    b = a + n;
    cols = reinterpret_cast<int*>(b + n);
  }
};

// A short global array (twiddles, the column list) staged through registers:
// with a compile-time length the loads are issued at the start of a kernel
// together with its other loads and written to LDS after the first wait,
// instead of a load-wait-write loop that costs a memory latency of its own.
template <class T, int NF, int NT>
struct Staged {
  static constexpr int K = NF > 0 ? (NF + NT - 1) / NT : 1;
  T v[K];
  // branch-free (lanes past n load element n - 1, never stored; of an empty
  // array, the element every buffer holds), so that the compiler's waits count
  // these loads exactly
  template <class A>
  __device__ __forceinline__ void load(A* src, int n) {
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = src[min(int(threadIdx.x) + k * NT, max(n - 1, 0))];
  }
  __device__ __forceinline__ void store(T* dst, int n) const {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int e = threadIdx.x + k * NT;
      if (e < n) dst[e] = v[k];
    }
  }
};
template <class T, int NF, int NT, class A>
__device__ __forceinline__ void copy_to_lds(T* dst, A* src, int n) {
  for (int e = threadIdx.x; e < n; e += NT) dst[e] = src[e];
}

// Row pass, forward.  Item = (slice, y * ngr + g): coil group g of image row
// y.  The groups of row y also perform the dual step of row y (TV or TGV),
// each on its own range of pixels.  Then for
// each coil of the group: S_c * src row -> ifftshift -> PE-FFT -> fftshift
// -> sampled columns -> T1 [c][y][ks].
// With ndual > 0 (a single slice, dense items) the dual step is left to
// ndual further workgroups after the nitems row items, each on a contiguous
// range of pixels (gap terms at part[nitems + b]), so that the FFT chains of
// the row items do not wait for it.
// The gap-evaluation variant holds extra FP64 accumulators; it is asked to
// fit five waves per SIMD, as many as the plain variant, so that the same
// tile shapes keep every block resident.
// Dual step (TV or TGV, MODE) of a single dense slice done by workgroups of
// their own, launched after the item workgroups of a pass: workgroup b of nd
// takes a contiguous pixel range, and the ranges go to XCDs in consecutive
// runs, so that the next row's pixels (forward differences) are mostly in
// the same L2.  Gap terms (GAP) to part[b].
template <class R, int MODE, bool GAP, int NT>
__device__ __forceinline__ void dual_workgroup(const SliceDev& d, int nd, double* part) {
  using C = Cx<R>;
  const int b = xcd_item(int(blockIdx.x) - int(gridDim.x) + nd, nd), W = d.W, WH = W * d.H;
  const int chunk = (WH + nd - 1) / nd;
  const int pa = min(WH, b * chunk), pe = min(WH, pa + chunk);
  const int k = gptr<int>(d.ctl)[CTL_ITER];
  const R sigma = R(d.sigma);
  const auto w0 = ball_any(sched_alpha<R>(d, d.alpha0, d.alpha0_end, k));
  const auto w1 = ball_any(sched_alpha<R>(d, d.alpha1, d.alpha1_end, k));
  const float rW = 1.0f / float(W);
  // GAP: the sums are formed as by 256 threads whatever NT is (wave w takes
  // the pixels of waves w, w + NT / 64, ... of those), so that every launch
  // that carries these workgroups finds the same bits.
  constexpr int VT = GAP ? kBlock : NT, VW = VT / 64, NW = NT / 64;
  __shared__ double red[GAP ? VW * kGapTerms : 1];
  const int lane = threadIdx.x & 63;
  for (int vw = threadIdx.x >> 6; vw < VW; vw += NW) {
    double t[kGapTerms] = {0};
    for (int i = pa + vw * 64 + lane; i < pe; i += VT) {
      const int y = qdiv(i, W, rW), x = i - y * W;
      dual_pixel<C, C, MODE == M_TGV, GAP>(d, x, y, sigma, w0, w1, t);
    }
    if (GAP) {
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        double v = t[k];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
        if (lane == 0) red[vw * kGapTerms + k] = v;
      }
    }
  }
  if (GAP) {
    __syncthreads();
    if (threadIdx.x < 3) {
      double v = 0;
      for (int w = 0; w < VW; ++w) v += red[w * kGapTerms + threadIdx.x];
      part[size_t(b) * kGapTerms + threadIdx.x] = v;
    }
  }
}

template <class R, int MODE, bool GAP, int NT, int NF>
__device__ __forceinline__ void rows_fwd(const SliceDev* sl, const int2* items, int nitems, int cb, double* part,
                                         int ndual, char* smem_raw) {
  using C = Cx<R>;
  if (int(blockIdx.x) >= nitems) {
    const SliceDev& d = sl[0];
    if constexpr (MODE == M_OP) {
      // operator forward: the output, of which the column pass writes the
      // listed columns only, is zeroed beside the row transforms
      const size_t n = size_t(d.W) * d.Hk * d.C, chunk = (n + ndual - 1) / ndual;
      const size_t b = size_t(blockIdx.x - nitems) * chunk, e = min(n, b + chunk);
      const auto out = gptr<C>(d.op_out);
      for (size_t i = b + threadIdx.x; i < e; i += NT) out[i] = pzero<C>();
    } else {
      if (!slice_active(d)) return;
      dual_workgroup<R, MODE, GAP, NT>(d, ndual, part + size_t(nitems) * kGapTerms);
    }
    return;
  }
  const int li = xcd_item(blockIdx.x, nitems);
  const int2 it = items ? items[li] : make_int2(0, li);  // null: the dense single-slice list
  const SliceDev& d = sl[it.x];
  const int W = NF > 0 ? NF : d.W, H = d.H, nc = d.ncols;
  const int y = it.y / d.ngr, g = it.y - y * d.ngr;
  const int c0 = g * cb, ncb = min(cb, d.C - c0);
  RowLds<C> L(smem_raw, W, cb);
  const auto gtw = gptr<const C>(d.planW.tw);
  const auto gcols = gptr<const int>(d.cols);
  Staged<C, NF, NT> s_tw;
  Staged<int, NF, NT> s_cols;
  if (NF > 0) {
    s_tw.load(gtw, W);
    s_cols.load(gcols, nc);
  } else {
    copy_to_lds<C, NF, NT>(L.tw, gtw, W);
    copy_to_lds<int, NF, NT>(L.cols, gcols, nc);
  }
  const auto src = gptr<const C>(MODE == M_OP ? d.op_in : d.ub) + size_t(y) * W;
  const auto S = gptr<const C>(d.S);
  const int G = W * d.Hk;
  const auto Sg = S ? S + size_t(c0) * G + size_t(y + d.y0) * W : S;  // coil c0, row y + y0
  const float rW = 1.0f / float(W), rnc = 1.0f / float(max(nc, 1));
  // With a compile-time length and at most kPrefetch elements per thread the
  // row and sensitivity values are loaded into registers first and combined
  // after the dual step, so that both sets of loads are in flight together.
  C ps[kPrefetch], pS[kPrefetch];
  const bool pf = NF > 0 && ncb * W <= kPrefetch * NT;
  if (pf) {
#pragma unroll
    for (int k = 0; k < kPrefetch; ++k) {
      const int e = threadIdx.x + k * NT;
      if (e < ncb * W) {
        const int cl = divn<NF>(e, W, rW), x = e - cl * W;
        ps[k] = src[x];
        if (S) pS[k] = Sg[cl * G + x];
      }
    }
  } else {
    for (int e = threadIdx.x; e < ncb * W; e += NT) {
      const int cl = divn<NF>(e, W, rW), x = e - cl * W;
      C z = src[x];
      if (S) z = z * Sg[cl * G + x];
      L.a[lp<NF>(cl * W + ishift_dst(x, W))] = z;
    }
  }
  // A finished slice's blocks leave before their first store; the check comes
  // after the loads above are issued, so its control-word load overlaps them.
  if (MODE != M_OP && !slice_active(d)) return;
  double t[kGapTerms] = {0};
  if (MODE != M_OP && ndual == 0) {
    // The dual step of row y is shared out over the row's coil groups in
    // pixel ranges of a multiple of 32, so no group carries all of it.
    const int chunk = ((W + d.ngr - 1) / d.ngr + 31) & ~31;
    const int xa = min(W, g * chunk), xe = min(W, xa + chunk);
    const int k = gptr<int>(d.ctl)[CTL_ITER];
    const R sigma = R(d.sigma);
    const R a0 = sched_alpha<R>(d, d.alpha0, d.alpha0_end, k);
    const R a1 = sched_alpha<R>(d, d.alpha1, d.alpha1_end, k);
    const auto w0 = ball_any(a0), w1 = ball_any(a1);
    for (int x = xa + threadIdx.x; x < xe; x += NT) dual_pixel<C, C, MODE == M_TGV, GAP>(d, x, y, sigma, w0, w1, t);
  }
  if (NF > 0) {
    s_tw.store(L.tw, W);
    s_cols.store(L.cols, nc);
  }
  if (pf) {
#pragma unroll
    for (int k = 0; k < kPrefetch; ++k) {
      const int e = threadIdx.x + k * NT;
      if (e < ncb * W) {
        const int cl = divn<NF>(e, W, rW), x = e - cl * W;
        L.a[lp<NF>(cl * W + ishift_dst(x, W))] = S ? ps[k] * pS[k] : ps[k];
      }
    }
  }
  __syncthreads();
  C* res = fft_n<R, NT, false, NF>(L.a, L.b, ncb, d.planW, L.tw);
  // T1 is row-major per coil, [c][y][ks], like T2: a row writes nc
  // contiguous entries per coil (the column pass gathers with a stride)
  const auto T1 = gptr<C>(d.T1) + (size_t(c0) * H + y) * nc;  // coil c0, row y
  for (int e = threadIdx.x; e < ncb * nc; e += NT) {
    const int cl = qdiv(e, nc, rnc), ks = e - cl * nc;
    T1[size_t(cl) * H * nc + ks] = res[lp<NF>(cl * W + fshift_src(L.cols[ks], W))];
  }
  if (GAP) block_sum<3, NT>(reinterpret_cast<double(&)[3]>(t), part + size_t(li) * kGapTerms);
}

template <class R, int MODE, bool GAP, int NT, int NF>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(GAP ? 5 : 1))) void k_rows_fwd(const SliceDev* sl, const int2* items, int nitems, int cb,
                                                 double* part, int ndual) {
  extern __shared__ char smem_raw[];
  rows_fwd<R, MODE, GAP, NT, NF>(sl, items, nitems, cb, part, ndual, smem_raw);
}

// The first launch of an operator application takes its descriptor by value
// and leaves it in memory for the launches after it (a launch or a copy less
// in front of it: 3.2 us and its gap).
__device__ __forceinline__ void store_desc(const SliceDev& d, SliceDev* dst) {
  static_assert(sizeof(SliceDev) % 8 == 0, "whole words");
  if (blockIdx.x == 0)
    for (int i = threadIdx.x; i < int(sizeof(SliceDev) / 8); i += blockDim.x)
      reinterpret_cast<uint64_t*>(dst)[i] = reinterpret_cast<const uint64_t*>(&d)[i];
}
template <class R, int NT, int NF>
__global__ __launch_bounds__(NT) void k_op_rows_fwd(const SliceDev d, SliceDev* dst, int nitems, int cb, int nzero) {
  extern __shared__ char smem_raw[];
  store_desc(d, dst);
  rows_fwd<R, M_OP, false, NT, NF>(&d, nullptr, nitems, cb, nullptr, nzero, smem_raw);
}

// Column pass.  CMODE: 0 solver (forward, r prox, adjoint), 1 operator
// forward (writes op_out {W, Hk, C}), 2 operator adjoint (reads op_in).
// PF (solver, compile-time length, at most kColPrefetchCols columns per
// item): the gather and the prox operands go through registers.  It is a
// template argument so that the other gather, a loop, is not compiled into
// the same kernel: the compiler's waits after the join of the two would count
// the prox loads as outstanding before the FFT.
enum { CM_SOLVE = 0, CM_FWD = 1, CM_ADJ = 2 };

// DUAL (M_TV or M_TGV; a single dense slice): ndual workgroups after the
// column items do the dual step of the iteration (dual_workgroup, gap terms
// to part_dual), which reads and writes none of what the column items do;
// with the adjoint row pass also writing the next T1 (k_rows_adj NEXT) an
// iteration is these two launches.
template <class R, int CMODE, bool GAP, int NT, int NF, bool PF, int DUAL>
__device__ __forceinline__ void cols(const SliceDev* sl, const int2* items, int nitems, int cg, double* part, int ndual,
                                     double* part_dual, char* smem_raw) {
  static_assert(!PF || (NF > 0 && CMODE == CM_SOLVE), "register prefetch needs a compile-time length");
  static_assert(DUAL == 0 || CMODE == CM_SOLVE, "dual workgroups: solver iterations");
  if (DUAL != 0 && int(blockIdx.x) >= nitems) {
    const SliceDev& d = sl[0];
    if (!slice_active(d)) return;
    dual_workgroup<R, DUAL, GAP, NT>(d, ndual, part_dual);
    return;
  }
  const int li = xcd_item(blockIdx.x, nitems);
  const int2 it = items ? items[li] : make_int2(0, li);  // null: the dense single-slice list
  const SliceDev& d = sl[it.x];
  using C = Cx<R>;
  const int W = d.W, H = d.H, Hk = NF > 0 ? NF : d.Hk, y0 = d.y0, nc = d.ncols;
  const int c = it.y / d.ngroups, g = it.y - c * d.ngroups;
  const int ks0 = g * cg, ncg = min(cg, nc - ks0);
  const R scale = R(1) / sqrt(R(W) * R(Hk));
  const auto Mc = gptr<const R>(d.Mc);
  C* tw = reinterpret_cast<C*>(smem_raw);
  C* bufA = tw + Hk;
  C* bufB = bufA + lds_pad(cg * Hk);
  const auto gtw = gptr<const C>(d.planH.tw);
  Staged<C, NF, NT> s_tw;
  if (NF > 0) s_tw.load(gtw, Hk);
  else copy_to_lds<C, NF, NT>(tw, gtw, Hk);
  const float rHk = 1.0f / float(Hk), rncg = 1.0f / float(ncg);
  C* res;
  double t[2] = {0, 0};
  // TGV_prox_r_kernel (tgv_kernels.cuh:212-223) operands; columns ks0.. of
  // coil c are contiguous in the compact layout.  With a compile-time length
  // they are loaded into registers, issued after the T1 gather: vector memory
  // loads return in issue order, so the gather's wait before the LDS stores
  // leaves them in flight, and they arrive during the forward FFT.
  const R sigma = R(d.sigma), lambda = R(d.lambda), inv_sl = rcp(R(1) + sigma * lambda);
  const auto fk = gptr<const C>(d.fk) + (size_t(c) * nc + ks0) * Hk;
  const auto rk = gptr<C>(d.rk) + (size_t(c) * nc + ks0) * Hk;
  const auto mk = Mc + size_t(ks0) * Hk;
  constexpr int KP = NF > 0 ? (kColPrefetchCols * NF + NT - 1) / NT : 1;
  C pf_f[KP], pf_r[KP];
  R pf_m[KP];
  constexpr bool pf = PF;
  // the gather of the zero-padded, ifftshifted columns of T1 (coil c, columns
  // ks0.., a stride of nc in y): into registers with a compile-time length
  const auto T1 = gptr<const C>(d.T1) + size_t(c) * H * nc + ks0;
  C pf_t[KP];
  if (pf) {
#pragma unroll
    for (int k = 0; k < KP; ++k) {
      const int e = threadIdx.x + k * NT;
      if (e < ncg * Hk) {
        const int j = qdiv(e, ncg, rncg), cl = e - j * ncg;
        const int yy = ishift_src(j, Hk) - y0;
        pf_t[k] = (yy >= 0 && yy < H) ? C(T1[yy * nc + cl]) : pzero<C>();
      }
    }
    // branch-free (lanes past the columns load the last element, unused), so
    // that the compiler's wait for the gather counts these loads as issued
    const int last = ncg * Hk - 1;
#pragma unroll
    for (int k = 0; k < KP; ++k) {
      const int e = min(int(threadIdx.x) + k * NT, last);
      pf_f[k] = fk[e];
      pf_r[k] = rk[e];
      pf_m[k] = mk[e];
    }
  }
  if (CMODE == CM_SOLVE && !slice_active(d)) return;  // after the loads are issued, before any store
  if (CMODE != CM_ADJ) {
    // registers -> LDS with the prefetch, else the gather straight into LDS
    if (pf) {
#pragma unroll
      for (int k = 0; k < KP; ++k) {
        const int e = threadIdx.x + k * NT;
        if (e < ncg * Hk) {
          const int j = qdiv(e, ncg, rncg), cl = e - j * ncg;
          bufA[lp<NF>(cl * Hk + j)] = pf_t[k];
        }
      }
    } else {
      for (int e = threadIdx.x; e < ncg * Hk; e += NT) {
        const int j = qdiv(e, ncg, rncg), cl = e - j * ncg;
        const int fe = ishift_src(j, Hk);
        const int yy = fe - y0;
        bufA[lp<NF>(cl * Hk + j)] = (yy >= 0 && yy < H) ? C(T1[yy * nc + cl]) : pzero<C>();
      }
    }
    if (NF > 0) s_tw.store(tw, Hk);
    __syncthreads();
    res = fft_n<R, NT, false, NF>(bufA, bufB, ncg, d.planH, tw);
    C* other = (res == bufA) ? bufB : bufA;
    if (CMODE == CM_FWD) {
      const auto out = gptr<C>(d.op_out);
      for (int e = threadIdx.x; e < ncg * Hk; e += NT) {
        const int cl = divn<NF>(e, Hk, rHk), kfe = e - cl * Hk;
        const R m = Mc[size_t(ks0 + cl) * Hk + kfe];
        out[(size_t(c) * Hk + kfe) * W + gptr<const int>(d.cols)[ks0 + cl]] = (m * scale) * res[lp<NF>(cl * Hk + fshift_src(kfe, Hk))];
      }
      return;
    }
    // prox of r on A ubar - f
    auto prox = [&](int e, R m, C f, C r) {
      const int cl = divn<NF>(e, Hk, rHk), kfe = e - cl * Hk;
      const C a = (m * scale) * res[lp<NF>(cl * Hk + fshift_src(kfe, Hk))];
      const C tmp = a - f;
      const C rn = (r + sigma * tmp) * inv_sl;
      rk[e] = rn;
      if (GAP) {
        t[0] += dabs2(tmp);
        t[1] += dabs2(tmp - lambda * rn);
      }
      other[lp<NF>(cl * Hk + ishift_dst(kfe, Hk))] = m * rn;
    };
    if (pf) {
#pragma unroll
      for (int k = 0; k < KP; ++k) {
        const int e = threadIdx.x + k * NT;
        if (e < ncg * Hk) prox(e, pf_m[k], pf_f[k], pf_r[k]);
      }
    } else {
      for (int e = threadIdx.x; e < ncg * Hk; e += NT) prox(e, mk[e], fk[e], rk[e]);
    }
    __syncthreads();
    res = fft_n<R, NT, true, NF>(other, res, ncg, d.planH, tw);
  } else {
    if (NF > 0) s_tw.store(tw, Hk);
    const auto in = gptr<const C>(d.op_in);
    for (int e = threadIdx.x; e < ncg * Hk; e += NT) {
      const int cl = divn<NF>(e, Hk, rHk), kfe = e - cl * Hk;
      const R m = Mc[size_t(ks0 + cl) * Hk + kfe];
      bufA[lp<NF>(cl * Hk + ishift_dst(kfe, Hk))] = m * in[(size_t(c) * Hk + kfe) * W + gptr<const int>(d.cols)[ks0 + cl]];
    }
    __syncthreads();
    res = fft_n<R, NT, true, NF>(bufA, bufB, ncg, d.planH, tw);
  }
  const auto T2 = gptr<C>(d.T2) + size_t(c) * H * nc + ks0;
  for (int e = threadIdx.x; e < ncg * H; e += NT) {
    const int yy = qdiv(e, ncg, rncg), cl = e - yy * ncg;
    T2[yy * nc + cl] = scale * res[lp<NF>(cl * Hk + fshift_src(yy + y0, Hk))];
  }
  if (GAP) block_sum<2, NT>(t, part + size_t(li) * kGapTerms);
}

template <class R, int CMODE, bool GAP, int NT, int NF, bool PF = false, int DUAL = 0>
__global__ __launch_bounds__(NT) void k_cols(const SliceDev* sl, const int2* items, int nitems, int cg,
                                             double* part, int ndual, double* part_dual) {
  extern __shared__ char smem_raw[];
  cols<R, CMODE, GAP, NT, NF, PF, DUAL>(sl, items, nitems, cg, part, ndual, part_dual, smem_raw);
}
template <class R, int NT, int NF>
__global__ __launch_bounds__(NT) void k_op_cols_adj(const SliceDev d, SliceDev* dst, int nitems, int cg) {
  extern __shared__ char smem_raw[];
  store_desc(d, dst);
  cols<R, CM_ADJ, false, NT, NF, false, 0>(&d, nullptr, nitems, cg, nullptr, 0, nullptr, smem_raw);
}

// Column pass of the lengths 8 M 8 (those of with_direct_cols): a thread does one
// butterfly of every stage, and what comes before the first stage, between the
// two transforms and after the last one stays in its registers.  The first
// stage reads T1; the last stage of the forward transform leaves outputs
// i + q n / 8 in a thread, which are the inputs of the first stage of the
// inverse transform, so the prox of those samples is done on registers; the
// last stage writes T2.  Four barriers and four passes through LDS, where the
// general kernel has eight and nine.
// Bound by this chain (descriptor, loads, six stages, stores) with every
// workgroup resident at once, not by its bytes: of a launch of 640 points with
// the dual step the vector instructions take 2.7 us and the waves wait 49 % of
// their time.  Per launch, general kernel before, this one after (kernel trace):
// 640 points, 15 coils x 80 columns with the dual step 12.1 -> 10.6 us; between
// events, in three passes, 768 points, 15 x 117 15.9 -> 13.1 and 512 points in
// double precision (a runtime plan before), 8 x 64 11.4 -> 7.5.
// At most CS columns per group (max_cg): two of 640 points (160 threads) were
// faster than three or four, 2 and 4 % of an iteration, and
// two of 512 in double than four.
template <class R, int NF>
struct ColShape {
  static constexpr int M = NF / 64, NR = NF / 8;  // middle radix; butterflies of a radix-8 stage
  static constexpr int CS = NR > 80 ? 2 : 160 / NR;  // columns at most
  static constexpr int NT = (CS * (NR > 64 ? NR : 64) + 63) / 64 * 64;
  static constexpr int NP = NF + NF / 8;          // LDS slots of a column, one pad slot per 8 elements
  static constexpr size_t lds = (NF + 2 * size_t(CS) * NP) * sizeof(Cx<R>);
};
template <class R, int CMODE, bool GAP, int NF, int DUAL>
__device__ __forceinline__ void cols_direct(const SliceDev* sl, const int2* items, int nitems, int cg, double* part,
                                            int ndual, double* part_dual, char* smem_raw) {
  using C = Cx<R>;
  using Sh = ColShape<R, NF>;
  constexpr int CS = Sh::CS, M = Sh::M, NR = Sh::NR, NT = Sh::NT, NP = Sh::NP, NRP = NR + NR / 8, Hk = NF;
  static_assert(NF == 64 * M && NR % 8 == 0, "8 M 8, padded");
  if (DUAL != 0 && int(blockIdx.x) >= nitems) {
    const SliceDev& d = sl[0];
    if (!slice_active(d)) return;
    dual_workgroup<R, DUAL, GAP, NT>(d, ndual, part_dual);
    return;
  }
  const int li = xcd_item(blockIdx.x, nitems);
  const int2 it = items ? items[li] : make_int2(0, li);  // null: the dense single-slice list
  const SliceDev& d = sl[it.x];
  const int W = d.W, H = d.H, y0 = d.y0, nc = d.ncols;
  const int c = it.y / d.ngroups, g = it.y - c * d.ngroups;
  const R scale = R(1) / sqrt(R(W) * R(Hk));
  const R sigma = R(d.sigma), lambda = R(d.lambda), inv_sl = rcp(R(1) + sigma * lambda);
  C* const tw = reinterpret_cast<C*>(smem_raw);
  C* const bufA = tw + Hk;
  C* const bufB = bufA + CS * NP;
  const auto T1 = gptr<const C>(d.T1) + size_t(c) * H * nc;
  const auto T2 = gptr<C>(d.T2) + size_t(c) * H * nc;
  const auto fk = gptr<const C>(d.fk) + size_t(c) * nc * Hk;
  const auto rk = gptr<C>(d.rk) + size_t(c) * nc * Hk;
  const auto Mc = gptr<const R>(d.Mc);
  const auto cols = gptr<const int>(d.cols);
  const auto in = gptr<const C>(d.op_in) + size_t(c) * Hk * W;
  const auto out = gptr<C>(d.op_out) + size_t(c) * Hk * W;
  // A thread's butterflies: the stages at T1 and T2 take columns fastest (the
  // columns of a row are contiguous there), the stages at the prox the i of a
  // column (f, r and the mask are contiguous along it), the middle stages one
  // column per wave.
  const int ca = threadIdx.x % CS, ia = threadIdx.x / CS;
  const int cp = threadIdx.x / NR, ip = threadIdx.x - cp * NR;
  const int cm = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), im = threadIdx.x & 63;
  double t[2] = {0, 0};
  Staged<C, NF, NT> s_tw;
  s_tw.load(gptr<const C>(d.planH.tw), Hk);
  // sample kfe of the transform's element i + q n / 8 (fftshift of an even length)
  auto kfe = [](int i, int q) { return i + NR * ((q + 4) & 7); };
  // radix-M stage of the middle: bufA -> bufB
  auto middle = [&](bool act, bool inv) {
    if (act) {
      const int kk = im & 7;
      const C* a = bufA + cm * NP + im + im / 8;
      C z[M];
      z[0] = a[0];
#pragma unroll
      for (int j = 1; j < M; ++j) z[j] = a[72 * j] * twd(tw, 8 * j * kk, inv);
      Dft<R, M>::run(z, inv ? R(1) : R(-1));
      C* b = bufB + cm * NP + (im / 8) * (9 * M) + kk;
#pragma unroll
      for (int q = 0; q < M; ++q) b[9 * q] = z[q];
    }
    __syncthreads();
  };
  const int ks0 = g * cg, ncs = min(cg, nc - ks0);
  const bool acta = ia < NR && ca < ncs, actp = cp < ncs, actm = cm < ncs;
  const int kp = ks0 + (actp ? cp : 0), e0 = kp * Hk + (actp ? ip : 0);
  C x[8], pf[8], pr[8];
  R pm[8];
  bool ok[8];
  // branch-free loads, so that the compiler's wait for the first ones counts
  // those after them (lanes without work and zero-padded rows load one valid
  // element, unused)
  if (CMODE != CM_ADJ) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int yy = kfe(ia, j) - y0;
      ok[j] = acta && yy >= 0 && yy < H;
      x[j] = T1[ok[j] ? yy * nc + ks0 + ca : 0];
    }
  }
  const int col = CMODE == CM_SOLVE ? 0 : int(cols[kp]);
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int e = e0 + kfe(0, q);
    pm[q] = Mc[e];
    if (CMODE == CM_SOLVE) {
      pf[q] = fk[e];
      pr[q] = rk[e];
    } else if (CMODE == CM_ADJ) {
      pf[q] = in[size_t((actp ? ip : 0) + kfe(0, q)) * W + col];
    }
  }
  if (CMODE == CM_SOLVE && !slice_active(d)) return;  // after the loads are issued, before any store
  s_tw.store(tw, Hk);
  if (CMODE != CM_ADJ) {
    // forward: 8, M, 8
    if (acta) {
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = csel(ok[j], x[j], pzero<C>());
      Dft<R, 8>::run(x, R(-1));
#pragma unroll
      for (int q = 0; q < 8; ++q) bufA[ca * NP + 9 * ia + q] = x[q];
    }
    __syncthreads();
    middle(actm, false);
    if (actp) {
      const C* b = bufB + cp * NP + ip + ip / 8;
      x[0] = b[0];
#pragma unroll
      for (int j = 1; j < 8; ++j) x[j] = b[j * NRP] * twd(tw, j * ip, false);
      Dft<R, 8>::run(x, R(-1));
    }
  }
  if (actp) {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      if (CMODE == CM_ADJ) {
        x[q] = pm[q] * pf[q];
        continue;
      }
      const C a = (pm[q] * scale) * x[q];
      if (CMODE == CM_FWD) {
        out[size_t(kfe(ip, q)) * W + col] = a;
        continue;
      }
      // prox of r on A ubar - f: TGV_prox_r_kernel (tgv_kernels.cuh:212-223)
      const C tmp = a - pf[q];
      const C rn = (pr[q] + sigma * tmp) * inv_sl;
      rk[e0 + kfe(0, q)] = rn;
      if (GAP) {
        t[0] += dabs2(tmp);
        t[1] += dabs2(tmp - lambda * rn);
      }
      x[q] = pm[q] * rn;
    }
    if (CMODE != CM_FWD) {
      // inverse: 8, M, 8
      Dft<R, 8>::run(x, R(1));
#pragma unroll
      for (int q = 0; q < 8; ++q) bufA[cp * NP + 9 * ip + q] = x[q];
    }
  }
  if (CMODE == CM_FWD) return;
  __syncthreads();
  middle(actm, true);
  if (acta) {
    const C* b = bufB + ca * NP + ia + ia / 8;
    x[0] = b[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) x[j] = b[j * NRP] * twd(tw, j * ia, true);
    Dft<R, 8>::run(x, R(1));
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int yy = kfe(ia, q) - y0;
      if (yy >= 0 && yy < H) T2[yy * nc + ks0 + ca] = scale * x[q];
    }
  }
  if (GAP) block_sum<2, NT>(t, part + size_t(li) * kGapTerms);
}

template <class R, int CMODE, bool GAP, int NF, int DUAL = 0>
__global__ __launch_bounds__((ColShape<R, NF>::NT)) void k_cols_direct(const SliceDev* sl, const int2* items, int nitems,
                                                                     int cg, double* part, int ndual,
                                                                     double* part_dual) {
  extern __shared__ char smem_raw[];
  cols_direct<R, CMODE, GAP, NF, DUAL>(sl, items, nitems, cg, part, ndual, part_dual, smem_raw);
}
template <class R, int NF>
__global__ __launch_bounds__((ColShape<R, NF>::NT)) void k_op_cols_adj_direct(const SliceDev d, SliceDev* dst, int nitems,
                                                                            int cg) {
  extern __shared__ char smem_raw[];
  store_desc(d, dst);
  cols_direct<R, CM_ADJ, false, NF, 0>(&d, nullptr, nitems, cg, nullptr, 0, nullptr, smem_raw);
}

// Primal step of pixel (x, y) given w = (A^* r)(x, y):
// TGV_primal_u_noprox_kernel (tgv_kernels.cuh:432-467) and, for TGV,
// TGV_primal_v_kernel (:647-686).  Adds |w - div p|^2 and |p + div_sym q|^2
// to t for the gap.
template <class R, int MODE, bool GAP>
__device__ __forceinline__ void mri_primal_pixel(const SliceDev& d, int x, int y, Cx<R> w, R tau, R theta,
                                                 double* t) {
  using C = Cx<R>;
  const int W = d.W, H = d.H;
  const size_t n = size_t(W) * H, i = size_t(y) * W + x;
  const auto u = gptr<C>(d.u);
  const auto ub = gptr<C>(d.ub);
  const auto px = gptr<const C>(d.p);
  const auto py = px + n;
  const C uo = u[i];
  const C div = dmx<C>(px, x, i, W) + dmy<C>(py, y, i, W, H);
  const C un = uo + tau * (div - w);
  u[i] = un;
  ub[i] = (R(1) + theta) * un - theta * uo;
  if (GAP) t[0] += dabs2(w - div);
  if (MODE == M_TGV) {
    const double rv = vstep_pixel<C, C>(d, x, y, tau, theta);
    if (GAP) t[1] += rv;
  }
}

// Register slots per thread of the adjoint row pass: the 1024-thread variant
// must stay within 64 VGPRs (two blocks per CU), so it holds fewer.
template <int NT> constexpr int rows_adj_ps() { return NT >= 1024 ? 6 : kPrefetch; }
template <int NT> constexpr int rows_adj_pt() { return NT >= 1024 ? 2 : 4; }
// The straight-line path loads its sensitivity slots unconditionally, so it
// is built for as many as it uses: 5 coils for each thread group (15 coils on
// rows of 320, 20 on rows of 256, 10 on rows of 384 and 512), and for the
// padded lengths of two groups also 8 (16 coils).  8 slots spill in every paired
// iteration, 6 registers (28 bytes) on rows of 384 and 21 (88 bytes) on rows of
// 512, where 5 spill 1 and 13: 10 coils on rows of 384 take 30.5 us per iteration
// with 8, 28 with 5; 12 coils 34 us, against 40 in three passes and
// k_mri_primal.
constexpr int kFusedSlots = 5, kFusedSlotsMore = 8;
constexpr bool fused_more_ok(int W) { return ct_pad_ok(W) && kRowAdjThreadsWide / W == 2; }
// Coils per thread group.
constexpr int fused_coils(int W, int C) {
  const int ngs = kRowAdjThreadsWide / W < C ? kRowAdjThreadsWide / W : C;
  return (C + ngs - 1) / ngs;
}
// Its LDS: twiddles, the coils' padded slots and the group sums (ct_pad_ok), or
// two unpadded buffers.  (15 coils on rows of 384: 61 KB, two workgroups per
// CU; with the 95 KB of two buffers one, and 28.7 us instead of 22.5.)
constexpr size_t fused_lds(int W, int C, size_t esize) {
  const int ngs = kRowAdjThreadsWide / W < C ? kRowAdjThreadsWide / W : C;
  return (ct_pad_ok(W) ? size_t(W) + size_t(C) * (W + W / 8) + size_t(ngs) * W : size_t(W) * (1 + 2 * size_t(C))) * esize;
}

// Element e of a wave-uniform base: a 32-bit byte offset, so that the access
// takes the base from scalar registers (fewer address instructions and
// registers).  The offset must stay below 4 GB.
template <class P>
__device__ __forceinline__ auto& at(P base, uint32_t e) {
  using T = std::remove_reference_t<decltype(*base)>;
  using Byte = std::conditional_t<std::is_const<T>::value, const char, char>;
  const auto b = (__attribute__((address_space(1))) Byte*)base;
  return *(P)(b + e * uint32_t(sizeof(T)));
}

// The adjoint row pass of one row y holding all coils (FUSED in k_rows_adj):
// T2 row -> ifftshift -> inverse PE-FFT -> fftshift -> * conj(S_c), summed
// over the coils (thread group gi takes coils [gi ch, (gi + 1) ch) of pixel
// gx, the group sums added in group order), then the u step of row y
// (TGV_primal_u_noprox_kernel, tgv_kernels.cuh:432-467).  Load order: the
// twiddles, the T2 gather, u and p of the primal step (their arithmetic
// waits for them), then the sensitivities, which the FFT does not need.
template <class R, int MODE, bool GAP, int NT, int NF, int PS, bool NEXT>
__device__ __forceinline__ void rows_adj_fused(const SliceDev& d, int y, double* part_rows, char* smem_raw) {
  using C = Cx<R>;
  constexpr int W = NF, PT = rows_adj_pt<NT>();
  // Lengths with the padded layout: one padded slot range per coil, whose
  // T2 scatter, transforms (fft_wave) and T1 entries one wavefront does
  // alone (coils wave, wave + NW, ...; lb holds the coil-group sums), so the
  // block waits at four barriers.  Other lengths: two unpadded buffers and
  // workgroup-wide stages (lp without padding is the identity for them).
  constexpr bool IP = ct_pad_ok(NF);
  constexpr int NW = NT / 64, NPW = W + W / 8;  // waves; padded slots per coil
  constexpr int SPW = (PS * (NT / NF) + NW - 1) / NW;  // coils per wave
  const int H = d.H, nc = d.ncols, ncb = d.C;
  const int ngs = min(NT / W, ncb), ch = (ncb + ngs - 1) / ngs;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  C* const tw = reinterpret_cast<C*>(smem_raw);
  C* const la = tw + W;
  C* const lb = la + (IP ? ncb * NPW : ncb * W);
  Staged<C, NF, NT> s_tw;
  s_tw.load(gptr<const C>(d.planW.tw), W);
  if constexpr (!IP)
    for (int e = threadIdx.x; e < ncb * W; e += NT) la[e] = pzero<C>();
  // T2 row y of every coil and the PE column of each sampled entry (padded
  // layout: entries ks = lane + 64 k of the wave's coils, branch-free with
  // clamped indices; else entry e = tid + k NT of the row)
  const float rnc = 1.0f / float(max(nc, 1));
  const auto T2 = gptr<const C>(d.T2) + size_t(y) * nc;
  const auto gcols = gptr<const int>(d.cols);
  const int cstride = H * nc, last = max(nc - 1, 0);
  C pT[IP ? SPW : 1][PT];
  int pK[PT];
  if constexpr (IP) {
#pragma unroll
    for (int k = 0; k < PT; ++k) pK[k] = at(gcols, uint32_t(min(lane + 64 * k, last)));
#pragma unroll
    for (int sq = 0; sq < SPW; ++sq)
#pragma unroll
      for (int k = 0; k < PT; ++k)
        pT[sq][k] = at(T2 + min(wave + NW * sq, ncb - 1) * cstride, uint32_t(min(lane + 64 * k, last)));
  } else {
#pragma unroll
    for (int k = 0; k < PT; ++k) {
      const int e = threadIdx.x + k * NT;
      if (e < ncb * nc) {
        const int cl = qdiv(e, nc, rnc), ks = e - cl * nc;
        pT[0][k] = T2[cl * cstride + ks];
        pK[k] = gcols[ks];
      }
    }
  }
  // u(x, y) and the neighbours of div p (p is final for this iteration),
  // loaded branch-free (threads past the row load pixel 0, unused)
  const R tau = R(d.tau), theta = R(d.theta);
  // (NEXT: every thread group takes the u step of its own pixel gx, each
  // forming the same values, so that its forward products need no exchange
  // of the new ubar through LDS)
  const int gi = threadIdx.x / W, gx = threadIdx.x - gi * W;
  const int x = threadIdx.x;
  const bool upix = NEXT ? gi < ngs : x < W;
  const int xr = NEXT ? (gi < ngs ? gx : 0) : (x < W ? x : 0);
  const size_t n = size_t(W) * H, row = size_t(y) * W;
  const auto pp = gptr<const C>(d.p) + row;
  const C e_uo = at(gptr<const C>(d.u) + row, uint32_t(xr));
  const C cx = at(pp, uint32_t(xr)), mx = at(pp, uint32_t(max(xr - 1, 0)));
  const C cy = at(pp + n, uint32_t(xr)), my = at(pp + n - (y > 0 ? W : 0), uint32_t(xr));
  // sensitivities, branch-free (spare slots load a valid element, unused)
  const int G = W * d.Hk;
  const auto Sg = gptr<const C>(d.S) + size_t(y + d.y0) * W;
  C pS[PS];
#pragma unroll
  for (int k = 0; k < PS; ++k) pS[k] = at(Sg, uint32_t(min(gi * ch + k, ncb - 1)) * uint32_t(G) + uint32_t(gx));
  if (!slice_active(d)) return;  // after the loads are issued, before any store
  // descriptor fields of the stores, read before the asm below (after it
  // the compiler no longer takes the descriptor for unmodified, and would
  // read them with vector loads at the end of the block)
  const auto gu = gptr<C>(d.u) + row;
  const auto gub = gptr<C>(d.ub) + row;
  const auto gctl = gptr<int>(d.ctl);
  const int row_beg = d.row_beg;
  // div p = dmx + dmy (the same operations as dmx / dmy), formed here: the
  // empty asm keeps the compiler from sinking it past the FFT, where the
  // four neighbours would hold registers instead of the one sum
  const C dx = csel(xr > 0, csel(xr < W - 1, cx - mx, -mx), cx);
  const C dy = csel(y > 0, csel(y < H - 1, cy - my, -my), cy);
  C e_div = dx + dy;
  asm volatile("" : "+v"(e_div.re), "+v"(e_div.im));
  C* res;
  C* other;
  if constexpr (IP) {
    // each wave: its coils' slots zeroed, their T2 entries at the
    // ifftshifted PE slots, then (twiddles in) their inverse transforms
#pragma unroll
    for (int sq = 0; sq < SPW; ++sq) {
      const int cl = wave + NW * sq;
      if (cl < ncb) {
        C* const sp = la + cl * NPW;
        for (int e = lane; e < NPW; e += 64) sp[e] = pzero<C>();
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int k = 0; k < PT; ++k) {
          const int j = ishift_dst(pK[k], W);
          if (lane + 64 * k < nc) sp[j + (j >> 3)] = pT[sq][k];
        }
        __builtin_amdgcn_wave_barrier();
      }
    }
    s_tw.store(tw, W);
    __syncthreads();  // twiddles
#pragma unroll
    for (int sq = 0; sq < SPW; ++sq) {
      const int cl = wave + NW * sq;
      if (cl < ncb) fft_wave<R, NF, 0, 1, true>(la + cl * NPW, tw);
    }
    res = la;
    other = lb;
  } else {
    s_tw.store(tw, W);
    __syncthreads();  // zero fill, twiddles
#pragma unroll
    for (int k = 0; k < PT; ++k) {
      const int e = threadIdx.x + k * NT;
      if (e < ncb * nc) {
        const int cl = qdiv(e, nc, rnc);
        la[lp<NF, false>(cl * W + ishift_dst(pK[k], W))] = pT[0][k];
      }
    }
    __syncthreads();
    res = fft_n<R, NT, true, NF, false>(la, lb, ncb, d.planW, tw);
    other = (res == la) ? lb : la;
  }
  __syncthreads();  // every coil's inverse transform (fft_n: its last stage's)
  if (gi < ngs) {
    C acc = pzero<C>();
#pragma unroll
    for (int k = 0; k < PS; ++k) {
      const int cl = gi * ch + k;
      if (k < ch && cl < ncb) acc = acc + mulconj(res[lp<NF, IP>(cl * W + fshift_src(gx, W))], pS[k]);
    }
    other[gi * W + gx] = acc;
  }
  __syncthreads();
  double t[2] = {0, 0};
  if (upix) {
    C w = other[xr];
    for (int q = 1; q < ngs; ++q) w = w + other[q * W + xr];
    const C un = e_uo + tau * (e_div - w);
    const C ubn = (R(1) + theta) * un - theta * e_uo;
    if (!NEXT || gi == 0) {  // (NEXT: one thread group stores and counts the pixel)
      at(gu, uint32_t(xr)) = un;
      at(gub, uint32_t(xr)) = ubn;
      if (GAP) t[0] += dabs2(w - e_div);
    }
    if constexpr (NEXT) {
      // the next forward row pass's input (what k_rows_fwd's row items form
      // from ubar, the same operations): S_c ubar, ifftshifted, into the
      // inverse transform's buffer (consumed above the barrier)
#pragma unroll
      for (int k = 0; k < PS; ++k) {
        const int cl = gi * ch + k;
        if (k < ch && cl < ncb) res[lp<NF, IP>(cl * W + ishift_dst(gx, W))] = ubn * pS[k];
      }
    }
  }
  if (GAP) block_sum<2, NT>(t, part_rows + size_t(row_beg + y) * kGapTerms);
  if (y == 0 && threadIdx.x == 0) {
    gctl[CTL_ITER] += 1;
    gctl[CTL_RUPD] += 1;
  }
  if constexpr (NEXT) {
    // The rest of the next iteration's forward row pass on the new ubar row:
    // PE-FFT -> fftshift -> the sampled columns -> T1 [c][y][ks] (the
    // entries of the T2 gather, in the same layout).
    __syncthreads();  // products in res; the coil sums in other are read
    const auto T1 = gptr<C>(d.T1) + size_t(y) * nc;
    if constexpr (IP) {
#pragma unroll
      for (int sq = 0; sq < SPW; ++sq) {
        const int cl = wave + NW * sq;
        if (cl < ncb) {
          C* const sp = res + cl * NPW;
          fft_wave<R, NF, 0, 1, false>(sp, tw);
#pragma unroll
          for (int k = 0; k < PT; ++k) {
            const int ks = lane + 64 * k, j = fshift_src(pK[k], W);
            if (ks < nc) at(T1 + cl * cstride, uint32_t(ks)) = sp[j + (j >> 3)];
          }
        }
      }
    } else {
      C* fres = fft_n<R, NT, false, NF, false>(res, other, ncb, d.planW, tw);
#pragma unroll
      for (int k = 0; k < PT; ++k) {
        const int e = threadIdx.x + k * NT;
        if (e < ncb * nc) {
          const int cl = qdiv(e, nc, rnc);
          T1[size_t(cl) * H * nc + (e - cl * nc)] = fres[lp<NF, false>(cl * W + fshift_src(pK[k], W))];
        }
      }
    }
  }
}

// Row pass, adjoint.  Item = (slice, y * ngr_a + g): for each coil of group g,
// T2 row -> ifftshift -> inverse PE-FFT -> fftshift -> * conj(S_c), summed
// over the group's coils in order.  With several coil groups (ngr_a > 1) the
// sum goes to wpart[g][y][x] and k_mri_primal completes the step; with one
// group the block holds all of (A^* r)(., y) and performs the primal step of
// row y itself (MODE M_OP: writes A^* r to op_out).  The 1024-thread
// variant on swz-permuted buffers is held to 64 VGPRs (its slot arithmetic
// would take more), so that two workgroups share a CU.
// FUSED (sensitivity slots per thread; host-checked, see rows_adj_fused_ok): a
// compile-time row length, one
// coil group per row holding every coil (the u step follows in the block),
// 2 W <= NT, the coil products in registers (every thread group's coils fit
// its slots), the T2 row in registers, sensitivities present, and no v step
// in the row blocks (TGV: separate workgroups).  That path is straight-line,
// so the compiler's waits can leave the sensitivity loads, issued after the
// T2 gather and the primal-step loads, in flight during the inverse FFT (the
// other paths' runtime branches make it wait for every load before it).
// NEXT (with FUSED): the row blocks also compute the next iteration's T1
// from their new ubar row, which k_rows_fwd's row items would otherwise do
// (rows_adj_fused).  Its gap-evaluation variant (one iteration in
// gap_every) is not held to 64 VGPRs: within them it spilled.
template <class R, int MODE, bool GAP, int NT, int NF, int FUSED = 0, bool NEXT = false>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(NT >= 1024 && NF > 0 && ct_pad_ok(NF) && !(GAP && NEXT) ? 8 : 1))) void k_rows_adj(const SliceDev* sl, const int2* items, int nitems, int cb,
                                                 double* part_rows, int nvstep) {
  extern __shared__ char smem_raw[];
  using C = Cx<R>;
  static_assert(FUSED == 0 || (NF > 0 && MODE != M_OP && NT == kRowAdjThreadsWide), "fused adjoint row path");
  static_assert(!NEXT || FUSED != 0, "next forward rows: the fused path");
  if (int(blockIdx.x) >= nitems) {
    // nvstep workgroups after the row items (a single slice): the v step of
    // TGV_primal_v_kernel on contiguous pixel ranges, where the row items
    // would do it before their FFT (gap terms at part_rows[row_beg + H + b]);
    // elsewhere they only write zero gap terms.
    const SliceDev& d = sl[0];
    if (!slice_active(d)) return;
    // consecutive pixel ranges on one XCD (backward differences of q)
    const int b = xcd_item(int(blockIdx.x) - nitems, nvstep), W = d.W, WH = W * d.H;
    double t[2] = {0, 0};
    if (MODE == M_TGV && NF > 0 && d.ngr_a == 1 && 2 * W <= NT) {
      const int chunk = (WH + nvstep - 1) / nvstep;
      const int pa = min(WH, b * chunk), pe = min(WH, pa + chunk);
      const R tau = R(d.tau), theta = R(d.theta);
      const float rW = 1.0f / float(W);
      for (int i = pa + threadIdx.x; i < pe; i += NT) {
        const int y = qdiv(i, W, rW), x = i - y * W;
        const double rv = vstep_pixel<C, C>(d, x, y, tau, theta);
        if (GAP) t[1] += rv;
      }
    }
    if (GAP) block_sum<2, NT>(t, part_rows + size_t(d.row_beg + d.H + b) * kGapTerms);
    return;
  }
  const int li = xcd_item(blockIdx.x, nitems);
  const int2 it = items ? items[li] : make_int2(0, li);  // null: the dense single-slice list
  const SliceDev& d = sl[it.x];
  if constexpr (FUSED != 0) {
    rows_adj_fused<R, MODE, GAP, NT, NF, FUSED, NEXT>(d, it.y, part_rows, smem_raw);
    return;
  }
  const int W = NF > 0 ? NF : d.W, H = d.H, nc = d.ncols;
  const int y = it.y / d.ngr_a, g = it.y - y * d.ngr_a;
  const int c0 = g * cb, ncb = min(cb, d.C - c0);
  // the wide variant keeps two blocks per CU only without the LDS padding
  constexpr bool LP = NT != kRowAdjThreadsWide;
  RowLds<C> L(smem_raw, W, cb, LP);
  const auto gtw = gptr<const C>(d.planW.tw);
  const auto gcols = gptr<const int>(d.cols);
  Staged<C, NF, NT> s_tw;
  if (NF > 0) s_tw.load(gtw, W);
  else copy_to_lds<C, NF, NT>(L.tw, gtw, W);
  for (int e = threadIdx.x; e < (LP ? lds_pad(ncb * W) : ncb * W); e += NT) L.a[e] = pzero<C>();
  const float rW = 1.0f / float(W), rnc = 1.0f / float(max(nc, 1));
  // sensitivities of the group's coils on row y + y0: with a compile-time
  // length loaded into registers before the T2 gather (one latency for both)
  const auto S = gptr<const C>(d.S);
  const int G = W * d.Hk;
  const auto Sg = S ? S + size_t(c0) * G + size_t(y + d.y0) * W : S;
  constexpr int PS = rows_adj_ps<NT>(), PT = rows_adj_pt<NT>();
  C pS[PS];
  // Coil sum in registers (one block holds the whole row, u step fused):
  // thread t = gi W + x takes pixel x of the coils [gi ch, (gi + 1) ch) of
  // the row, multiplies and sums them after the FFT, and the ng partial sums
  // of a pixel are added in group order.  Otherwise every thread takes
  // elements e = cl W + x in turn and one thread per pixel sums all coils.
  const int ngs = min(NT / W, ncb), ch = (ncb + ngs - 1) / max(ngs, 1);
  const bool gsum = NF > 0 && Sg && MODE != M_OP && d.ngr_a == 1 && 2 * W <= NT && ch <= PS;
  const int gi = threadIdx.x / W, gx = threadIdx.x - gi * W;
  if (gsum) {
#pragma unroll
    for (int k = 0; k < PS; ++k) {
      const int cl = gi * ch + k;
      if (gi < ngs && k < ch && cl < ncb) pS[k] = Sg[cl * G + gx];
    }
  }
  const bool pf = !gsum && NF > 0 && Sg && ncb * W <= PS * NT;
  if (pf) {
#pragma unroll
    for (int k = 0; k < PS; ++k) {
      const int e = threadIdx.x + k * NT;
      if (e < ncb * W) {
        const int cl = divn<NF>(e, W, rW), x = e - cl * W;
        pS[k] = Sg[cl * G + x];
      }
    }
  }
  // the T2 gather (values and their PE columns) into registers with a
  // compile-time length, issued with the sensitivity loads
  const auto T2 = gptr<const C>(d.T2) + (size_t(c0) * H + y) * nc;  // row y of coil c0
  const int cstride = H * nc;
  C pT[PT];
  int pK[PT];
  const bool pft = NF > 0 && ncb * nc <= PT * NT;
  if (pft) {
#pragma unroll
    for (int k = 0; k < PT; ++k) {
      const int e = threadIdx.x + k * NT;
      if (e < ncb * nc) {
        const int cl = qdiv(e, nc, rnc), ks = e - cl * nc;
        pT[k] = T2[cl * cstride + ks];
        pK[k] = gcols[ks];
      }
    }
  } else {
    copy_to_lds<int, NF, NT>(L.cols, gcols, nc);
  }
  if (MODE != M_OP && !slice_active(d)) return;  // after the loads above are issued, before any store
  // With all coils of the row in one block of at least 2 W threads, the
  // parts of the primal step that do not need A^* r run before the FFT, so
  // their loads overlap those of S and T2: threads x < W load u(x, y) and
  // form div p (p is final for this iteration), threads W + x perform the
  // whole v step of pixel x (TGV_primal_v_kernel, tgv_kernels.cuh:647-686,
  // needs only p and q).
  const R tau = R(d.tau), theta = R(d.theta);
  double t[2] = {0, 0};
  const bool early = NF > 0 && MODE != M_OP && d.ngr_a == 1 && 2 * W <= NT;
  C e_uo = pzero<C>(), e_div = pzero<C>();
  if (early) {
    const int x = threadIdx.x;
    if (x < W) {
      const size_t n = size_t(W) * H, i = size_t(y) * W + x;
      const auto px = gptr<const C>(d.p);
      e_uo = gptr<const C>(d.u)[i];
      e_div = dmx<C>(px, x, i, W) + dmy<C>(px + n, y, i, W, H);
    } else if (MODE == M_TGV && nvstep == 0 && x < 2 * W) {
      const double rv = vstep_pixel<C, C>(d, x - W, y, tau, theta);
      if (GAP) t[1] += rv;
    }
  }
  if (NF > 0) s_tw.store(L.tw, W);
  __syncthreads();  // zero fill, twiddles, column list
  if (pft) {
#pragma unroll
    for (int k = 0; k < PT; ++k) {
      const int e = threadIdx.x + k * NT;
      if (e < ncb * nc) {
        const int cl = qdiv(e, nc, rnc);
        L.a[lp<NF, LP>(cl * W + ishift_dst(pK[k], W))] = pT[k];
      }
    }
  } else {
    for (int e = threadIdx.x; e < ncb * nc; e += NT) {
      const int cl = qdiv(e, nc, rnc), ks = e - cl * nc;
      L.a[lp<NF, LP>(cl * W + ishift_dst(L.cols[ks], W))] = T2[cl * cstride + ks];
    }
  }
  __syncthreads();
  C* res = fft_n<R, NT, true, NF, LP>(L.a, L.b, ncb, d.planW, L.tw);
  C* other = (res == L.a) ? L.b : L.a;
  if (gsum) {
    if (gi < ngs) {
      C acc = pzero<C>();
#pragma unroll
      for (int k = 0; k < PS; ++k) {
        const int cl = gi * ch + k;
        if (k < ch && cl < ncb) acc = acc + mulconj(res[lp<NF, LP>(cl * W + fshift_src(gx, W))], pS[k]);
      }
      other[gi * W + gx] = acc;
    }
  } else if (pf) {
#pragma unroll
    for (int k = 0; k < PS; ++k) {
      const int e = threadIdx.x + k * NT;
      if (e < ncb * W) {
        const int cl = divn<NF>(e, W, rW), x = e - cl * W;
        other[lp<NF, LP>(cl * W + x)] = mulconj(res[lp<NF, LP>(cl * W + fshift_src(x, W))], pS[k]);
      }
    }
  } else {
    for (int e = threadIdx.x; e < ncb * W; e += NT) {
      const int cl = divn<NF>(e, W, rW), x = e - cl * W;
      const C v = res[lp<NF, LP>(cl * W + fshift_src(x, W))];
      other[lp<NF, LP>(cl * W + x)] = Sg ? mulconj(v, Sg[cl * G + x]) : v;
    }
  }
  __syncthreads();
  if (d.ngr_a > 1) {
    const auto wp = gptr<C>(d.wpart) + (size_t(g) * H + y) * W;
    for (int x = threadIdx.x; x < W; x += NT) {
      C acc = other[lp<NF, LP>(x)];
      for (int cl = 1; cl < ncb; ++cl) acc = acc + other[lp<NF, LP>(cl * W + x)];
      wp[x] = acc;
    }
    return;
  }
  if (early) {
    const int x = threadIdx.x;
    if (x < W) {
      C w;
      if (gsum) {
        w = other[x];
        for (int q = 1; q < ngs; ++q) w = w + other[q * W + x];
      } else {
        w = other[lp<NF, LP>(x)];
        for (int cl = 1; cl < ncb; ++cl) w = w + other[lp<NF, LP>(cl * W + x)];
      }
      const size_t i = size_t(y) * W + x;
      const C un = e_uo + tau * (e_div - w);
      gptr<C>(d.u)[i] = un;
      gptr<C>(d.ub)[i] = (R(1) + theta) * un - theta * e_uo;
      if (GAP) t[0] += dabs2(w - e_div);
    }
  } else {
    for (int x = threadIdx.x; x < W; x += NT) {
      C w = other[lp<NF, LP>(x)];
      for (int cl = 1; cl < ncb; ++cl) w = w + other[lp<NF, LP>(cl * W + x)];
      if (MODE == M_OP) gptr<C>(d.op_out)[size_t(y) * W + x] = w;
      else mri_primal_pixel<R, MODE, GAP>(d, x, y, w, tau, theta, t);
    }
  }
  if (MODE == M_OP) return;
  if (GAP) block_sum<2, NT>(t, part_rows + size_t(d.row_beg + y) * kGapTerms);
  if (y == 0 && threadIdx.x == 0) {
    gptr<int>(d.ctl)[CTL_ITER] += 1;
    gptr<int>(d.ctl)[CTL_RUPD] += 1;
  }
}

// Primal half of the MRI solvers for slices with several coil groups:
// w = sum_g wpart[g] (A^* r), then the primal step of each pixel.
// Item = (slice, first row), rpi rows; the block is sized to cover them in
// one pass (all loads of a thread issued together).  MODE M_OP writes w to
// op_out instead (operator adjoint).  Slices with one coil group are done in
// k_rows_adj.
template <class R, int MODE, bool GAP>
__global__ __launch_bounds__(1024) void k_mri_primal(const SliceDev* sl, const int2* items, int nitems, int rpi,
                                                     double* part) {
  const int li = xcd_item(blockIdx.x, nitems);
  const int2 it = items ? items[li] : make_int2(0, li * rpi);  // null: the dense single-slice list
  const SliceDev& d = sl[it.x];
  if ((MODE != M_OP && !slice_active(d)) || d.ngr_a == 1) return;
  using C = Cx<R>;
  const int W = d.W, H = d.H, ngr = d.ngr_a;
  const size_t n = size_t(W) * H;
  const int ya = it.y, yb = min(H, ya + rpi);
  const auto wp = gptr<const C>(d.wpart);
  const R tau = R(d.tau), theta = R(d.theta);
  double t[2] = {0, 0};
  const int cnt = (yb - ya) * W;
  for (int idx = threadIdx.x; idx < cnt; idx += blockDim.x) {
    const int yy = idx / W;
    const int x = idx - yy * W, y = ya + yy;
    const size_t i = size_t(y) * W + x;
    C w = wp[i];
    for (int g = 1; g < ngr; ++g) w = w + wp[size_t(g) * n + i];
    if (MODE == M_OP) gptr<C>(d.op_out)[i] = w;
    else mri_primal_pixel<R, MODE, GAP>(d, x, y, w, tau, theta, t);
  }
  if (MODE == M_OP) return;
  if (GAP) block_sum_dyn<2>(t, part + size_t(li) * kGapTerms);
  if (ya == 0 && threadIdx.x == 0) {
    gptr<int>(d.ctl)[CTL_ITER] += 1;
    gptr<int>(d.ctl)[CTL_RUPD] += 1;
  }
}

// ---------------------------------------------------------------------------
// Gap reduction: one block per slice, fixed summation order.
// Denoising: part[0] dual, part[1] primal, part[2] restore1, part[3] restore2
// over the row items.  MRI: part[0] rows_fwd, part[2] rows_adj over the row
// items, part[1] cols over the column items.
// ---------------------------------------------------------------------------
constexpr int kGapThreads = kBlock;  // one workgroup per slice (1024 threads measured slower)

template <class R>
__global__ __launch_bounds__(kGapThreads) void k_gap_reduce(const SliceDev* sl, int kind, const double* p0,
                                                       const double* p1, const double* p2,
                                                       const double* p3) {
  const SliceDev& d = sl[blockIdx.x];
  if (!slice_active(d)) return;
  const bool mri = kind == K_TGV_MRI || kind == K_TV_OP || kind == K_TGV_OP;
  double s[kGapTerms] = {0};
  double mx = 0;
  if (mri) {
    // four items per step, their loads issued before the additions (which
    // keep the order of a plain strided loop)
    for (int i0 = d.rg_beg + threadIdx.x; i0 < d.rg_end; i0 += 4 * kGapThreads) {
      double a[4][3];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int i = i0 + u * kGapThreads;
        const bool in = i < d.rg_end;
        const double* q = p0 + size_t(in ? i : i0) * kGapTerms;
        a[u][0] = in ? q[0] : 0.0;
        a[u][1] = in ? q[1] : 0.0;
        a[u][2] = in ? q[2] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        s[0] += a[u][0];
        s[1] += a[u][1];
        s[2] += a[u][2];
      }
    }
  }
  for (int i = d.row_beg + threadIdx.x; i < d.row_end; i += kGapThreads) {
    const double* a = p0 + size_t(i) * kGapTerms;
    if (kind == K_TV) {
      s[0] += a[0];
      s[1] += a[3];
      s[2] += p1[size_t(i) * kGapTerms + 0];
      s[3] += p1[size_t(i) * kGapTerms + 1];
    } else if (kind == K_TGV) {
      s[0] += a[0];
      s[1] += a[1];
      s[2] += a[3];
      mx = fmax(mx, p2[size_t(i) * kGapTerms + 0]);
      s[4] += p3[size_t(i) * kGapTerms + 0];
      s[5] += p3[size_t(i) * kGapTerms + 1];
    } else {
      s[5] += p2[size_t(i) * kGapTerms + 0];
      s[6] += p2[size_t(i) * kGapTerms + 1];
    }
  }
  if (mri) {
    for (int i0 = d.col_beg + threadIdx.x; i0 < d.col_end; i0 += 4 * kGapThreads) {
      double a[4][2];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int i = i0 + u * kGapThreads;
        const bool in = i < d.col_end;
        const double* q = p1 + size_t(in ? i : i0) * kGapTerms;
        a[u][0] = in ? q[0] : 0.0;
        a[u][1] = in ? q[1] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        s[3] += a[u][0];
        s[4] += a[u][1];
      }
    }
  }
  __shared__ double tot[kGapTerms];
  block_sum<kGapTerms, kGapThreads>(s, tot);
  if (kind == K_TGV) mx = block_max<kGapThreads>(mx);
  __syncthreads();
  if (threadIdx.x != 0) return;
  const double lam = d.lambda;
  double P = 0, D = 0, c0 = 0, c1 = 0, c2 = 0;
  if (kind == K_TV) {
    // ROF: P(ubar) = sum|grad ubar| + lambda/2 ||ubar - f||^2,
    //      D(p) = -Re<div p, f> - ||div p||^2 / (2 lambda).
    P = tot[0] + 0.5 * lam * tot[1];
    D = -tot[2] - tot[3] / (2.0 * lam);
  } else if (kind == K_TGV) {
    P = d.alpha1 * tot[0] + d.alpha0 * tot[1] + 0.5 * lam * tot[2];
    const double a = tot[4], b = tot[5];
    const double smax = mx > 0 ? fmin(1.0, d.alpha1 / mx) : 1.0;
    const double so = b > 0 ? fmin(fmax(lam * a / b, 0.0), smax) : smax;
    D = so * a - so * so * b / (2.0 * lam);
    c0 = mx;
  } else {
    // Partial gap on the ball of radius (rho_u, rho_v) around (ubar, vbar):
    // sum of Fenchel-Young gaps plus rho * stationarity residuals.
    const int k = gptr<int>(d.ctl)[CTL_ITER] - 1;
    const bool tgv = kind != K_TV_OP;
    const double a0 = tgv ? double(sched_alpha<R>(d, d.alpha0, d.alpha0_end, k)) : 0.0;
    const double a1 = tgv ? double(sched_alpha<R>(d, d.alpha1, d.alpha1_end, k)) : 1.0;
    const double bk = pow(1.0 + d.sigma * lam, -double(gptr<int>(d.ctl)[CTL_RUPD]));
    const double preg = a1 * tot[0] + a0 * tot[1];
    P = (tot[3] + d.F0) / (2.0 * lam) + preg;
    const double fy = (tot[4] + d.F0 * bk * bk) / (2.0 * lam) + preg - tot[2];
    c1 = sqrt(tot[5]);
    c2 = sqrt(tot[6]);
    const double G = fy + d.radius_u * c1 + (tgv ? d.radius_v * c2 : 0.0);
    D = P - G;
    c0 = fy;
  }
  const double rel = (P - D) / fmax(fabs(P), 1e-300);
  d.stats[ST_P] = P;
  d.stats[ST_D] = D;
  d.stats[ST_GAP] = P - D;
  d.stats[ST_REL] = rel;
  d.stats[ST_C0] = c0;
  d.stats[ST_C1] = c1;
  d.stats[ST_C2] = c2;
  gptr<int>(d.ctl)[CTL_NGAP] += 1;
  if (d.gap_tol > 0 && rel <= d.gap_tol) {
    gptr<int>(d.ctl)[CTL_ACTIVE] = 0;
    gptr<int>(d.ctl)[CTL_DONE_AT] = gptr<int>(d.ctl)[CTL_ITER];
  }
}

// ---------------------------------------------------------------------------
// Setup kernels
// ---------------------------------------------------------------------------
// Gather f {W, Hk, C} into [c][ks][kfe], zero r; one block per (slice, c, kfe
// row) item given as (slice, c * Hk + kfe).  Writes |f|^2 over unlisted
// columns of that row to part.
template <class R>
__global__ __launch_bounds__(kBlock) void k_compact(const SliceDev* sl, const int2* items, const void* f_full,
                                                    double* part) {
  const int2 it = items[blockIdx.x];
  const SliceDev& d = sl[it.x];
  using C = Cx<R>;
  const int W = d.W, Hk = d.Hk, nc = d.ncols;
  const int c = it.y / Hk, kfe = it.y - c * Hk;
  const auto f = gptr<const C>(f_full) + (size_t(c) * Hk + kfe) * W;
  const auto fk = gptr<C>(d.fk);
  const auto rk = gptr<C>(d.rk);
  double t[1] = {0};
  for (int kx = threadIdx.x; kx < W; kx += kBlock) {
    const int ks = gptr<const int>(d.colmap)[kx];
    const C v = f[kx];
    if (ks >= 0) {
      const size_t idx = (size_t(c) * nc + ks) * Hk + kfe;
      fk[idx] = v;
      rk[idx] = pzero<C>();
    } else {
      t[0] += dabs2(v);
    }
  }
  block_sum<1>(t, part + size_t(blockIdx.x) * kGapTerms);
}

__global__ __launch_bounds__(kBlock) void k_zero(uint32_t* p, size_t n) {
  for (size_t i = size_t(blockIdx.x) * kBlock + threadIdx.x; i < n; i += size_t(gridDim.x) * kBlock) p[i] = 0u;
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
#define PDT_LAUNCH(kern, grid, lds, st, ...) hipLaunchKernelGGL(kern, dim3(grid), dim3(kBlock), lds, st, __VA_ARGS__)

// LDS of a CU on gfx950, its allocation granule, and an upper bound on the
// static LDS of any kernel here (block reductions).
constexpr size_t kLdsPerCu = 160 * 1024, kLdsGranule = 512, kStaticLdsMax = 2048;

size_t lds_occupancy(size_t need, int wpc, size_t limit) {
  if (wpc <= 0) return need;
  // wpc workgroups of `share` bytes fit, wpc + 1 do not (wpc <= 6, so the
  // static part's slack cannot let a further one in)
  const size_t share = (kLdsPerCu / size_t(wpc)) / kLdsGranule * kLdsGranule;
  if (share <= kStaticLdsMax) return need;
  const size_t want = share - kStaticLdsMax;
  return want > limit ? need : (want > need ? want : need);
}

size_t lds_rows_bytes(int dtype, int cb, int W, int nc, bool padded) {
  const size_t e = (dtype == DT_C128 || dtype == DT_F64) ? 16 : 8;
  return (size_t(W) + 2 * size_t(padded ? lds_pad(cb * W) : cb * W)) * e + size_t(nc) * sizeof(int);
}
size_t lds_cols_bytes(int dtype, int cg, int Hk) {
  const size_t e = (dtype == DT_C128 || dtype == DT_F64) ? 16 : 8;
  return (size_t(Hk) + 2 * size_t(lds_pad(cg * Hk))) * e;
}

int num_stages(int kind) { return (kind == K_TV || kind == K_TGV) ? 2 : 4; }

const char* stage_name(int kind, int stage) {
  switch (kind) {
    case K_TV: return stage == 0 ? "k_tv_dual" : "k_tv_primal";
    case K_TGV: return stage == 0 ? "k_tgv_primal" : "k_tgv_dual";
    default: return stage == 0 ? "k_rows_fwd" : stage == 1 ? "k_cols" : stage == 2 ? "k_rows_adj" : "k_mri_primal";
  }
}

// Denoising stages: TV = {dual, primal}; TGV = {primal, dual (+ restoration
// on gap iterations)}.
template <class P, class S>
static void denoise_stage(const Launch& L, int kind, bool gap, int stage) {
  const int n = L.nrows;
  if (n == 0) return;
  const int2* rows = L.dense ? nullptr : L.rows;
  // occupancy cap: LDS only reserved (the kernels use none dynamically),
  // within the 64 KiB a launch may ask for without a raised attribute
  const size_t lds = lds_occupancy(0, L.wpc[WPC_DEN], 64 * 1024);
  // the half-iteration kernels with L.den_threads threads per workgroup
  auto launch = [&](auto nt) {
    constexpr int NT = decltype(nt)::value;
    if (kind == K_TV) {
      if (stage == 0) {
        if (gap) hipLaunchKernelGGL((k_tv_dual<P, true, NT>), dim3(n), dim3(NT), lds, L.stream, L.sl, rows, L.rpi, L.part[0]);
        else hipLaunchKernelGGL((k_tv_dual<P, false, NT>), dim3(n), dim3(NT), lds, L.stream, L.sl, rows, L.rpi, L.part[0]);
      } else {
        if (gap) hipLaunchKernelGGL((k_tv_primal<P, true, NT>), dim3(n), dim3(NT), lds, L.stream, L.sl, rows, L.rpi, L.part[1]);
        else hipLaunchKernelGGL((k_tv_primal<P, false, NT>), dim3(n), dim3(NT), lds, L.stream, L.sl, rows, L.rpi, L.part[1]);
      }
    } else if (stage == 0) {
      hipLaunchKernelGGL((k_tgv_primal<P, S, NT>), dim3(n), dim3(NT), lds, L.stream, L.sl, rows, L.rpi);
    } else if (L.den_pair) {
      // two pixels per thread: half the threads of the one-pixel launch (at least 256)
      constexpr int NP = NT > kBlock ? NT / 2 : kBlock;
      if (gap) hipLaunchKernelGGL((k_tgv_dual2<P, S, true, NP>), dim3(n), dim3(NP), lds, L.stream, L.sl, rows, L.rpi, L.part[0]);
      else hipLaunchKernelGGL((k_tgv_dual2<P, S, false, NP>), dim3(n), dim3(NP), lds, L.stream, L.sl, rows, L.rpi, L.part[0]);
    } else if (gap) {
      hipLaunchKernelGGL((k_tgv_dual<P, S, true, NT>), dim3(n), dim3(NT), lds, L.stream, L.sl, rows, L.rpi, L.part[0]);
    } else {
      hipLaunchKernelGGL((k_tgv_dual<P, S, false, NT>), dim3(n), dim3(NT), lds, L.stream, L.sl, rows, L.rpi, L.part[0]);
    }
  };
  if (L.den_threads >= 1024) launch(std::integral_constant<int, 1024>{});
  else if (L.den_threads >= 512) launch(std::integral_constant<int, 512>{});
  else launch(std::integral_constant<int, kBlock>{});
  if (kind == K_TGV && stage == 1 && gap) {
    PDT_LAUNCH((k_tgv_restore1<P, S>), n, 0, L.stream, L.sl, rows, L.rpi, L.part[2]);
    PDT_LAUNCH((k_tgv_restore2<P>), n, 0, L.stream, L.sl, rows, L.rpi, L.part[3]);
  }
}

#define PDT_LAUNCH_NT(kern, grid, nt, lds, st, ...) \
  hipLaunchKernelGGL(kern, dim3(grid), dim3(nt), lds, st, __VA_ARGS__)

// FFT lengths with kernels built on a compile-time plan (single precision; in
// double precision only the column pass of with_direct_cols); any other launch
// uses the runtime plan.
constexpr int kFftLengths[] = {256, 320, 368, 384, 512, 640, 736, 768};

// Calls fn(std::integral_constant<int, NF>) with NF = n when n has a
// compile-time plan for R, else NF = 0.
template <class R, class Fn>
static void with_fft_len(int n, Fn&& fn) {
  if constexpr (std::is_same<R, float>::value) {
    switch (n) {
      case 256: fn(std::integral_constant<int, 256>{}); return;
      case 320: fn(std::integral_constant<int, 320>{}); return;
      case 368: fn(std::integral_constant<int, 368>{}); return;
      case 384: fn(std::integral_constant<int, 384>{}); return;
      case 512: fn(std::integral_constant<int, 512>{}); return;
      case 640: fn(std::integral_constant<int, 640>{}); return;
      case 736: fn(std::integral_constant<int, 736>{}); return;
      case 768: fn(std::integral_constant<int, 768>{}); return;
      default: break;
    }
  }
  fn(std::integral_constant<int, 0>{});
}

// with_fft_len for the column lengths without k_cols_direct (N = 0: the
// runtime plan, for any length).
template <class R, class Fn>
static void with_other_len(int n, Fn&& fn) {
  if constexpr (std::is_same<R, float>::value) {
    if (n == 256) return fn(std::integral_constant<int, 256>{});
    if (n == 368) return fn(std::integral_constant<int, 368>{});
    if (n == 736) return fn(std::integral_constant<int, 736>{});
  }
  fn(std::integral_constant<int, 0>{});
}

// Calls fn(std::integral_constant<int, N>) when columns of n have k_cols_direct.
// Not for 256 points in single precision, where the general kernel is the
// faster one: it spreads two columns over 256 threads, which leaves each less to
// do one after the other.  us per launch, general against direct: 8 coils, 256
// columns wide 4.53 against 4.97; 20 coils with the dual step 6.91 against 7.38;
// an iteration of 256 x 256, 8 coils 12.5 against 13.0, 20 coils 17.4 against
// 18.2.  In double precision (no other compile-time plan) direct is the faster.
template <class R, class Fn>
static bool with_direct_cols(int n, Fn&& fn) {
  if constexpr (!std::is_same<R, float>::value) {
    if (n == 256) {
      fn(std::integral_constant<int, 256>{});
      return true;
    }
  }
  switch (n) {
    case 320: fn(std::integral_constant<int, 320>{}); return true;
    case 384: fn(std::integral_constant<int, 384>{}); return true;
    case 512: fn(std::integral_constant<int, 512>{}); return true;
    case 640: fn(std::integral_constant<int, 640>{}); return true;
    case 768: fn(std::integral_constant<int, 768>{}); return true;
    default: return false;
  }
}

bool fft_len_compiled(int dtype, int n) {
  if (dtype != DT_C64 && dtype != DT_F32) return false;
  for (int m : kFftLengths)
    if (m == n) return true;
  return false;
}

bool rows_adj_fused_ok(int dtype, int W, int C, int nc) {
  constexpr int NW = kRowAdjThreadsWide;
  // (a mask without listed columns has no T2 row to hold in registers)
  if (!fft_len_compiled(dtype, W) || 2 * W > NW || C < 1 || nc < 1) return false;
  // (unpadded lengths run their stages workgroup-wide, which takes work for
  // 1024 threads: 368 x 368, 3 coils 34.9 us per iteration this way, 32.8 not)
  if (!ct_pad_ok(W) && C * W < 8 * kRowThreads) return false;
  const int ch = fused_coils(W, C);
  // (padded lengths: a wave holds the listed columns of its coils, 64 per slot)
  const bool cols_fit = ct_pad_ok(W) ? nc <= 64 * rows_adj_pt<NW>() : C * nc <= rows_adj_pt<NW>() * NW;
  return ch <= (fused_more_ok(W) ? kFusedSlotsMore : kFusedSlots) && cols_fit;
}

// Calls fn with the sensitivity slots of the fused adjoint row path for C coils.
template <int NF, class Fn>
static void with_slots(int C, Fn&& fn) {
  if constexpr (fused_more_ok(NF)) {
    if (fused_coils(NF, C) > kFusedSlots) return fn(std::integral_constant<int, kFusedSlotsMore>{});
  }
  fn(std::integral_constant<int, kFusedSlots>{});
}

// Adjoint row pass with L.adj_threads threads per block (kRowThreads, or
// kRowAdjThreadsWide for items holding many coils).
template <class R, int MODE, int NF>
static void launch_rows_adj(const Launch& L, bool gap) {
  constexpr int NR = kRowThreads, NW = kRowAdjThreadsWide;
  const size_t lds = lds_occupancy(L.lds_rows_a, L.wpc[WPC_ADJ], init_kernel_attrs());
  if (L.adj_threads == NW) {
    const int nv = L.dense ? L.nvstep : 0;
    if constexpr (NF > 0 && MODE != M_OP) {
      if (L.adj_fused) {
        const size_t lds = lds_occupancy(fused_lds(NF, L.cb_a, sizeof(Cx<R>)), L.wpc[WPC_ADJ], init_kernel_attrs());
        with_slots<NF>(L.cb_a, [&](auto ps) {
          constexpr int PS = decltype(ps)::value;
          if (gap) PDT_LAUNCH_NT((k_rows_adj<R, MODE, true, NW, NF, PS>), L.nrg_a + nv, NW, lds, L.stream, L.sl, L.dense ? nullptr : L.rowgroups_a, L.nrg_a, L.cb_a, L.gap_rows, nv);
          else PDT_LAUNCH_NT((k_rows_adj<R, MODE, false, NW, NF, PS>), L.nrg_a + nv, NW, lds, L.stream, L.sl, L.dense ? nullptr : L.rowgroups_a, L.nrg_a, L.cb_a, L.gap_rows, nv);
        });
        return;
      }
    }
    if (gap) PDT_LAUNCH_NT((k_rows_adj<R, MODE, true, NW, NF>), L.nrg_a + nv, NW, lds, L.stream, L.sl, L.dense ? nullptr : L.rowgroups_a, L.nrg_a, L.cb_a, L.gap_rows, nv);
    else PDT_LAUNCH_NT((k_rows_adj<R, MODE, false, NW, NF>), L.nrg_a + nv, NW, lds, L.stream, L.sl, L.dense ? nullptr : L.rowgroups_a, L.nrg_a, L.cb_a, L.gap_rows, nv);
  } else {
    if (gap) PDT_LAUNCH_NT((k_rows_adj<R, MODE, true, NR, NF>), L.nrg_a, NR, lds, L.stream, L.sl, L.dense ? nullptr : L.rowgroups_a, L.nrg_a, L.cb_a, L.gap_rows, 0);
    else PDT_LAUNCH_NT((k_rows_adj<R, MODE, false, NR, NF>), L.nrg_a, NR, lds, L.stream, L.sl, L.dense ? nullptr : L.rowgroups_a, L.nrg_a, L.cb_a, L.gap_rows, 0);
  }
}

// Two on rows without a compile-time plan, in single precision and wherever
// one_group holds (double, 320 x 320, 15 coils, not one_group 74 us per iteration
// against 73 with four), while the items of two and the dual step's workgroups
// fit the chip's 2048 places for workgroups of 256 threads: up to about 1800
// items (1200 in double precision, whose registers leave fewer places).  Above,
// four are faster: us per iteration with two and four, 128 x 230, 20 coils (1280
// items of two) 36.2 and 37.9; 320 x 64, 12 coils (1920) 20.8 and 18.5; 320 x 200,
// 20 coils (3200) 35.7 and 32.7.  Where cb is the adjoint row pass's number too
// (not one_group), fours must fit by their LDS as well: 256 x 300, 20 coils 44.2
// and 36.8, 256 x 500, 16 coils (1024 items of four, 1024 places) 51.7 and 49.0,
// 225 x 500, 20 coils (1125) 63.6 and 72.8; with six or more per CU they need
// not, 400 x 270, 20 coils 1.08 times faster.  Measured at 982 sizes from 64 x 48
// to 400 x 700: in single precision and with one_group the rule's choice is at
// the worst 11 % off the better one, 0.4 % in the mean.  In double precision
// without one_group four stay the default everywhere, 6 % off in the mean (320 x
// 400, 6 coils 66.0 and 47.3 with two).
int default_cb(int dtype, int W, int H, int C, int nc, bool one_group) {
  if (fft_len_compiled(dtype, W)) return kDefaultCb;
  const long twos = long(H) * ((C + 1) / 2), fours = long(H) * ((C + 3) / 4);
  if (dtype == DT_C128) return one_group && twos <= 1200 ? 2 : kDefaultCb;
  if (twos <= 1800) return 2;
  if (one_group) return kDefaultCb;
  constexpr size_t kGranule = 1280;  // LDS is given out in these units
  const size_t lds = (lds_rows_bytes(dtype, kDefaultCb, W, nc) + kGranule - 1) / kGranule * kGranule;
  const long per_cu = long(kLdsMax / lds);
  return per_cu >= 6 || fours <= 256 * per_cu ? kDefaultCb : 2;
}

// Columns that a group of k_cols_direct holds at most; 0: not its length.
static int direct_cols(int dtype, int Hk) {
  int cs = 0;
  if (dtype == DT_C64) with_direct_cols<float>(Hk, [&](auto nf) { cs = ColShape<float, decltype(nf)::value>::CS; });
  else with_direct_cols<double>(Hk, [&](auto nf) { cs = ColShape<double, decltype(nf)::value>::CS; });
  return cs;
}

int max_cg(int dtype, int Hk, int nc) {
  int cg = nc > 1 ? nc : 1;
  if (const int cs = direct_cols(dtype, Hk)) cg = std::min(cg, cs);
  while (cg > 1 && lds_cols_bytes(dtype, cg, Hk) > init_kernel_attrs()) --cg;
  return cg;
}
int default_cg(int dtype, int Hk) {
  const int cs = direct_cols(dtype, Hk);
  return cs ? cs : 2;
}

// Column pass (DUAL: with the dual step's workgroups, gap terms to pd).
template <class R, int CMODE, bool GAP, int DUAL>
static void launch_cols(const Launch& L, const int2* items, int ndual, double* pd) {
  constexpr int NC = kColThreads;
  const size_t limit = init_kernel_attrs();
  bool done = false;
  with_direct_cols<R>(L.fft_h, [&](auto nf) {
    constexpr int NF = decltype(nf)::value;
    using Sh = ColShape<R, NF>;
    if (Sh::lds > limit) return;  // (a runtime that refuses more than 64 KB)
    done = true;
    PDT_LAUNCH_NT((k_cols_direct<R, CMODE, GAP, NF, DUAL>), L.ncolitems + ndual, Sh::NT, lds_occupancy(Sh::lds, L.wpc[WPC_COLS], limit), L.stream, L.sl, items, L.ncolitems, L.cg, L.part[1], ndual, pd);
  });
  if (done) return;
  const size_t lds = lds_occupancy(L.lds_cols, L.wpc[WPC_COLS], limit);
  with_other_len<R>(L.fft_h, [&](auto nf) {
    constexpr int NF = decltype(nf)::value;
    if constexpr (NF > 0 && CMODE == CM_SOLVE) {
      if (L.cg <= kColPrefetchCols) {
        PDT_LAUNCH_NT((k_cols<R, CMODE, GAP, NC, NF, true, DUAL>), L.ncolitems + ndual, NC, lds, L.stream, L.sl, items, L.ncolitems, L.cg, L.part[1], ndual, pd);
        return;
      }
    }
    PDT_LAUNCH_NT((k_cols<R, CMODE, GAP, NC, NF, false, DUAL>), L.ncolitems + ndual, NC, lds, L.stream, L.sl, items, L.ncolitems, L.cg, L.part[1], ndual, pd);
  });
}
// MRI stages: 0 rows_fwd, 1 cols, 2 rows_adj, 3 primal.  The FFT kernels are
// picked by L.fft_w (row length) and L.fft_h (column length).
template <class R, int MODE>
static void mri_stage_m(const Launch& L, bool gap, int stage) {
  constexpr int NR = kRowThreads;
  if (stage == 0) {
    const size_t lds = lds_occupancy(L.lds_rows, L.wpc[WPC_FWD], init_kernel_attrs());
    with_fft_len<R>(L.fft_w, [&](auto nf) {
      constexpr int NF = decltype(nf)::value;
      const int nd = L.dense ? L.ndual : 0;
      if (gap) PDT_LAUNCH_NT((k_rows_fwd<R, MODE, true, NR, NF>), L.nrg + nd, NR, lds, L.stream, L.sl, L.dense ? nullptr : L.rowgroups, L.nrg, L.cb, L.part[0], nd);
      else PDT_LAUNCH_NT((k_rows_fwd<R, MODE, false, NR, NF>), L.nrg + nd, NR, lds, L.stream, L.sl, L.dense ? nullptr : L.rowgroups, L.nrg, L.cb, L.part[0], nd);
    });
  } else if (stage == 1) {
    if (L.ncolitems == 0) return;
    const int2* items = L.dense ? nullptr : L.cols;
    if (gap) launch_cols<R, CM_SOLVE, true, 0>(L, items, 0, nullptr);
    else launch_cols<R, CM_SOLVE, false, 0>(L, items, 0, nullptr);
  } else if (stage == 2) {
    with_fft_len<R>(L.fft_w, [&](auto nf) {
      constexpr int NF = decltype(nf)::value;
      launch_rows_adj<R, MODE, NF>(L, gap);
    });
  } else {
    if (!L.split_primal) return;
    if (gap) PDT_LAUNCH_NT((k_mri_primal<R, MODE, true>), L.nrows, L.primal_threads, 0, L.stream, L.sl, L.rows, L.nrows, L.rpi, L.part[2]);
    else PDT_LAUNCH_NT((k_mri_primal<R, MODE, false>), L.nrows, L.primal_threads, 0, L.stream, L.sl, L.rows, L.nrows, L.rpi, L.part[2]);
  }
}

template <class R>
static void mri_stage(const Launch& L, int kind, bool gap, int stage) {
  if (kind == K_TV_OP) mri_stage_m<R, M_TV>(L, gap, stage);
  else mri_stage_m<R, M_TGV>(L, gap, stage);
}

// The two launches of a paired iteration (L.pair): 0 the column pass with
// the dual step's workgroups, 1 the fused adjoint row pass that also writes
// the next T1.  With the gap evaluation the partial sums go where the three
// passes put them: the dual step's after the forward row items' (which a
// paired iteration does not run; the engine zeroes theirs once), the column
// items' and the row items' as in those passes.
template <class R, int MODE, bool GAP>
static void mri_pair_m(const Launch& L, int which) {
  constexpr int NW = kRowAdjThreadsWide;
  if (which == 0) {
    launch_cols<R, CM_SOLVE, GAP, MODE>(L, nullptr, L.ndual, L.part[0] + size_t(L.nrg) * kGapTerms);
  } else {
    with_fft_len<R>(L.fft_w, [&](auto nf) {
      constexpr int NF = decltype(nf)::value;
      if constexpr (NF > 0) {
        const size_t lds = lds_occupancy(fused_lds(NF, L.cb_a, sizeof(Cx<R>)), L.wpc[WPC_ADJ], init_kernel_attrs());
        with_slots<NF>(L.cb_a, [&](auto ps) {
          PDT_LAUNCH_NT((k_rows_adj<R, MODE, GAP, NW, NF, decltype(ps)::value, true>), L.nrg_a + L.nvstep, NW, lds, L.stream, L.sl, nullptr, L.nrg_a, L.cb_a, L.gap_rows, L.nvstep);
        });
      }
    });
  }
}

void run_pair_stage(const Launch& L, int kind, int dtype, int which, bool gap) {
  if (dtype != DT_C64) return;  // pairs need the compile-time row plans (single precision)
  if (kind == K_TV_OP) {
    if (gap) mri_pair_m<float, M_TV, true>(L, which);
    else mri_pair_m<float, M_TV, false>(L, which);
  } else {
    if (gap) mri_pair_m<float, M_TGV, true>(L, which);
    else mri_pair_m<float, M_TGV, false>(L, which);
  }
}

void run_stage(const Launch& L, int kind, int dtype, bool fp16, bool gap, int stage) {
  if (kind == K_TV || kind == K_TGV) {
    switch (dtype) {
      case DT_F32:
        if (fp16) denoise_stage<float, _Float16>(L, kind, gap, stage);
        else denoise_stage<float, float>(L, kind, gap, stage);
        break;
      case DT_C64:
        if (fp16) denoise_stage<Cx<float>, Cx<_Float16>>(L, kind, gap, stage);
        else denoise_stage<Cx<float>, Cx<float>>(L, kind, gap, stage);
        break;
      case DT_F64: denoise_stage<double, double>(L, kind, gap, stage); break;
      case DT_C128: denoise_stage<Cx<double>, Cx<double>>(L, kind, gap, stage); break;
    }
  } else {
    if (dtype == DT_C64) mri_stage<float>(L, kind, gap, stage);
    else mri_stage<double>(L, kind, gap, stage);
  }
}

void run_iteration(const Launch& L, int kind, int dtype, bool fp16, bool gap) {
  for (int s = 0; s < num_stages(kind); ++s) run_stage(L, kind, dtype, fp16, gap, s);
}

void run_gap_reduce(const Launch& L, int kind, int dtype) {
  if (dtype == DT_F32 || dtype == DT_C64)
    hipLaunchKernelGGL((k_gap_reduce<float>), dim3(L.nsl), dim3(kGapThreads), 0, L.stream, L.sl, kind, L.part[0],
                       L.part[1], L.part[2], L.part[3]);
  else
    hipLaunchKernelGGL((k_gap_reduce<double>), dim3(L.nsl), dim3(kGapThreads), 0, L.stream, L.sl, kind, L.part[0],
                       L.part[1], L.part[2], L.part[3]);
}

template <class R>
static void op_forward(const Launch& L, const SliceDev& d) {
  constexpr int NR = kRowThreads;
  SliceDev* const dst = const_cast<SliceDev*>(L.sl);
  // zeroing workgroups: 32 elements per thread.  An output that overlaps the
  // input is zeroed before the row transforms read it, not beside them.
  const size_t in = size_t(d.W) * d.H, out = size_t(d.W) * d.Hk * d.C;
  const auto x = static_cast<const Cx<R>*>(d.op_in);
  const auto y = static_cast<const Cx<R>*>(d.op_out);
  const bool overlap = std::less<>()(x, y + out) && std::less<>()(y, x + in);
  if (overlap) run_zero(L.stream, d.op_out, out * sizeof(Cx<R>));
  const int nz = overlap ? 0 : int((out + 32 * NR - 1) / (32 * NR));
  with_fft_len<R>(L.fft_w, [&](auto nf) {
    PDT_LAUNCH_NT((k_op_rows_fwd<R, NR, decltype(nf)::value>), L.nrg + nz, NR, L.lds_rows, L.stream, d, dst, L.nrg, L.cb, nz);
  });
  launch_cols<R, CM_FWD, false, 0>(L, nullptr, 0, nullptr);
}

template <class R>
static void op_adjoint(const Launch& L, const SliceDev& d) {
  SliceDev* const dst = const_cast<SliceDev*>(L.sl);
  bool done = false;
  with_direct_cols<R>(L.fft_h, [&](auto nf) {
    constexpr int NF = decltype(nf)::value;
    using Sh = ColShape<R, NF>;
    if (Sh::lds > init_kernel_attrs()) return;
    done = true;
    PDT_LAUNCH_NT((k_op_cols_adj_direct<R, NF>), L.ncolitems, Sh::NT, Sh::lds, L.stream, d, dst, L.ncolitems, L.cg);
  });
  if (!done)
    with_other_len<R>(L.fft_h, [&](auto nf) {
      PDT_LAUNCH_NT((k_op_cols_adj<R, kColThreads, decltype(nf)::value>), L.ncolitems, kColThreads, L.lds_cols, L.stream, d, dst, L.ncolitems, L.cg);
    });
  with_fft_len<R>(L.fft_w, [&](auto nf) {
    constexpr int NF = decltype(nf)::value;
    launch_rows_adj<R, M_OP, NF>(L, false);
  });
  if (L.split_primal)
    PDT_LAUNCH_NT((k_mri_primal<R, M_OP, false>), L.nrows, L.primal_threads, 0, L.stream, L.sl, L.rows, L.nrows, L.rpi, L.part[2]);
}

// Raises the dynamic LDS limit of every FFT kernel instantiation to b bytes.
template <class R>
static bool set_lds_attrs(int b) {
  constexpr int NR = kRowThreads, NC = kColThreads;
  bool ok = true;
  auto set = [&](const void* f) {
    ok = ok && hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, b) == hipSuccess;
  };
  auto one = [&](auto nf) {
    constexpr int NF = decltype(nf)::value;
    set((const void*)&k_op_rows_fwd<R, NR, NF>);
    set((const void*)&k_rows_fwd<R, M_TV, false, NR, NF>);
    set((const void*)&k_rows_fwd<R, M_TV, true, NR, NF>);
    set((const void*)&k_rows_fwd<R, M_TGV, false, NR, NF>);
    set((const void*)&k_rows_fwd<R, M_TGV, true, NR, NF>);
    set((const void*)&k_rows_adj<R, M_OP, false, NR, NF>);
    set((const void*)&k_rows_adj<R, M_TV, false, NR, NF>);
    set((const void*)&k_rows_adj<R, M_TV, true, NR, NF>);
    set((const void*)&k_rows_adj<R, M_TGV, false, NR, NF>);
    set((const void*)&k_rows_adj<R, M_TGV, true, NR, NF>);
    set((const void*)&k_rows_adj<R, M_OP, false, kRowAdjThreadsWide, NF>);
    set((const void*)&k_rows_adj<R, M_TV, false, kRowAdjThreadsWide, NF>);
    set((const void*)&k_rows_adj<R, M_TV, true, kRowAdjThreadsWide, NF>);
    set((const void*)&k_rows_adj<R, M_TGV, false, kRowAdjThreadsWide, NF>);
    set((const void*)&k_rows_adj<R, M_TGV, true, kRowAdjThreadsWide, NF>);
    if constexpr (NF > 0) {
      auto fused = [&](auto ps) {
        constexpr int PS = decltype(ps)::value;
        set((const void*)&k_rows_adj<R, M_TV, false, kRowAdjThreadsWide, NF, PS>);
        set((const void*)&k_rows_adj<R, M_TV, true, kRowAdjThreadsWide, NF, PS>);
        set((const void*)&k_rows_adj<R, M_TGV, false, kRowAdjThreadsWide, NF, PS>);
        set((const void*)&k_rows_adj<R, M_TGV, true, kRowAdjThreadsWide, NF, PS>);
        set((const void*)&k_rows_adj<R, M_TV, false, kRowAdjThreadsWide, NF, PS, true>);
        set((const void*)&k_rows_adj<R, M_TGV, false, kRowAdjThreadsWide, NF, PS, true>);
        set((const void*)&k_rows_adj<R, M_TV, true, kRowAdjThreadsWide, NF, PS, true>);
        set((const void*)&k_rows_adj<R, M_TGV, true, kRowAdjThreadsWide, NF, PS, true>);
      };
      fused(std::integral_constant<int, kFusedSlots>{});
      if constexpr (fused_more_ok(NF)) fused(std::integral_constant<int, kFusedSlotsMore>{});
    }
  };
  auto col = [&](auto nf) {
    constexpr int NF = decltype(nf)::value;
    set((const void*)&k_cols<R, CM_SOLVE, false, NC, NF>);
    set((const void*)&k_cols<R, CM_SOLVE, true, NC, NF>);
    set((const void*)&k_cols<R, CM_FWD, false, NC, NF>);
    set((const void*)&k_op_cols_adj<R, NC, NF>);
    if constexpr (std::is_same<R, float>::value) {
      set((const void*)&k_cols<R, CM_SOLVE, false, NC, NF, false, M_TV>);
      set((const void*)&k_cols<R, CM_SOLVE, false, NC, NF, false, M_TGV>);
      set((const void*)&k_cols<R, CM_SOLVE, true, NC, NF, false, M_TV>);
      set((const void*)&k_cols<R, CM_SOLVE, true, NC, NF, false, M_TGV>);
    }
    if constexpr (NF > 0) {
      set((const void*)&k_cols<R, CM_SOLVE, false, NC, NF, true>);
      set((const void*)&k_cols<R, CM_SOLVE, true, NC, NF, true>);
      set((const void*)&k_cols<R, CM_SOLVE, false, NC, NF, true, M_TV>);
      set((const void*)&k_cols<R, CM_SOLVE, false, NC, NF, true, M_TGV>);
      set((const void*)&k_cols<R, CM_SOLVE, true, NC, NF, true, M_TV>);
      set((const void*)&k_cols<R, CM_SOLVE, true, NC, NF, true, M_TGV>);
    }
  };
  auto direct = [&](auto nf) {
    constexpr int NF = decltype(nf)::value;
    set((const void*)&k_cols_direct<R, CM_SOLVE, false, NF>);
    set((const void*)&k_cols_direct<R, CM_SOLVE, true, NF>);
    set((const void*)&k_cols_direct<R, CM_FWD, false, NF>);
    set((const void*)&k_op_cols_adj_direct<R, NF>);
    if constexpr (std::is_same<R, float>::value) {
      set((const void*)&k_cols_direct<R, CM_SOLVE, false, NF, M_TV>);
      set((const void*)&k_cols_direct<R, CM_SOLVE, false, NF, M_TGV>);
      set((const void*)&k_cols_direct<R, CM_SOLVE, true, NF, M_TV>);
      set((const void*)&k_cols_direct<R, CM_SOLVE, true, NF, M_TGV>);
    }
  };
  for (int n : kFftLengths) {
    with_direct_cols<R>(n, direct);
    with_other_len<R>(n, col);  // (0 for other lengths)
  }
  with_fft_len<R>(0, one);
  for (int n : kFftLengths)
    if (std::is_same<R, float>::value) with_fft_len<R>(n, one);
  return ok;
}

size_t init_kernel_attrs() {
  static size_t budget = 0;
  if (budget) return budget;
  // the block reductions use up to 2 KiB of static LDS
  const size_t want = kLdsMax - 4096;
  if (set_lds_attrs<float>(int(want)) && set_lds_attrs<double>(int(want))) {
    budget = want;
  } else {
    budget = 64 * 1024 - 4096;
  }
  (void)hipGetLastError();  // a refused attribute must not surface at the next launch check
  return budget;
}

void run_op_forward(const Launch& L, int dtype, const SliceDev& d) {
  if (dtype == DT_C64) op_forward<float>(L, d);
  else op_forward<double>(L, d);
}

void run_op_adjoint(const Launch& L, int dtype, const SliceDev& d) {
  if (dtype == DT_C64) op_adjoint<float>(L, d);
  else op_adjoint<double>(L, d);
}

int run_compact_data(const Launch& L, int dtype, const void* f_full, double* f0_part) {
  // L.rows here holds (slice, c * Hk + kfe) items
  if (dtype == DT_C64)
    PDT_LAUNCH((k_compact<float>), L.nrows, 0, L.stream, L.sl, L.rows, f_full, f0_part);
  else
    PDT_LAUNCH((k_compact<double>), L.nrows, 0, L.stream, L.sl, L.rows, f_full, f0_part);
  return L.nrows;
}

// Single-block reductions for set-up quantities, in a fixed order (each
// thread sums a strided subsequence, then a tree over the block): out[0] =
// sum_i a[i * stride] for i < n, and out[0] = sum_i |z_i|^2 over n pixels.
__device__ __forceinline__ void tree_sum_1024(double v, double* out) {
  __shared__ double red[1024];
  red[threadIdx.x] = v;
  __syncthreads();
  for (int o = 512; o > 0; o >>= 1) {
    if (int(threadIdx.x) < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = red[0];
}
// (Eight strided elements per step, loaded before they are added in order.)
__global__ __launch_bounds__(1024) void k_sum_strided(const double* a, int n, int stride, double* out) {
  double v = 0;
  for (int i0 = threadIdx.x; i0 < n; i0 += 8 * 1024) {
    double x[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = i0 + u * 1024;
      x[u] = i < n ? a[size_t(i) * stride] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) v += x[u];
  }
  tree_sum_1024(v, out);
}
template <class R>
__global__ __launch_bounds__(1024) void k_sumsq(const Cx<R>* z, int64_t n, double* out) {
  double v = 0;
  for (int64_t i0 = threadIdx.x; i0 < n; i0 += 8 * 1024) {
    Cx<R> x[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int64_t i = i0 + u * 1024;
      x[u] = i < n ? z[i] : pzero<Cx<R>>();
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) v += dabs2(x[u]);
  }
  tree_sum_1024(v, out);
}

void run_sum_strided(hipStream_t st, const double* a, int n, int stride, double* out) {
  PDT_LAUNCH_NT(k_sum_strided, 1, 1024, 0, st, a, n, stride, out);
}
void run_sumsq(hipStream_t st, int dtype, const void* z, int64_t n, double* out) {
  if (dtype == DT_C128) PDT_LAUNCH_NT((k_sumsq<double>), 1, 1024, 0, st, static_cast<const Cx<double>*>(z), n, out);
  else PDT_LAUNCH_NT((k_sumsq<float>), 1, 1024, 0, st, static_cast<const Cx<float>*>(z), n, out);
}

// Scratch of the allocation-free operator application: one array per GPU,
// part of the code object (no allocation), held until the process ends.
// Host code never passes the array's name to a kernel or a copy (on the host
// it is a stand-in, not a device address); it uses the per-device address
// that hipGetSymbolAddress returns, taken once per device with that device
// current.
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

void* noalloc_scratch(int device) {
  static std::mutex mu;
  static void* addr[kMaxDevices] = {};
  if (device < 0 || device >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lk(mu);
  if (!addr[device]) {
    int cur = -1;
    if (hipGetDevice(&cur) != hipSuccess || cur != device) return nullptr;
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess) return nullptr;
    addr[device] = p;
  }
  return addr[device];
}

void run_zero(hipStream_t st, void* ptr, size_t bytes) {
  const size_t n = bytes / 4;
  if (n == 0) return;
  size_t blocks = (n + kBlock - 1) / kBlock;
  if (blocks > 4096) blocks = 4096;
  PDT_LAUNCH(k_zero, blocks, 0, st, static_cast<uint32_t*>(ptr), n);
}

}  // namespace pdt
