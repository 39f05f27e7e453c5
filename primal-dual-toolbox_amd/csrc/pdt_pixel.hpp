// pdt_pixel.hpp -- device code shared by the kernel files: pixel arithmetic,
// storage types, address spaces, and the dual step of one pixel.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "pdt_desc.hpp"

namespace pdt {

// ---------------------------------------------------------------------------
// Pixel arithmetic
// ---------------------------------------------------------------------------
template <class R>
struct alignas(2 * sizeof(R)) Cx {
  R re, im;
};

template <class R> __device__ __forceinline__ Cx<R> operator+(Cx<R> a, Cx<R> b) { return {a.re + b.re, a.im + b.im}; }
template <class R> __device__ __forceinline__ Cx<R> operator-(Cx<R> a, Cx<R> b) { return {a.re - b.re, a.im - b.im}; }
template <class R> __device__ __forceinline__ Cx<R> operator-(Cx<R> a) { return {-a.re, -a.im}; }
// Complex products with explicit fused multiply-adds: left to the compiler,
// the contraction of a.re b.im + a.im b.re fused one product in one kernel
// and the other in another (both are one rounding short of two), so the same
// product of the same values differed in the last bit between kernels.
template <class R> __device__ __forceinline__ Cx<R> operator*(Cx<R> a, Cx<R> b) {
  return {fma(a.re, b.re, -(a.im * b.im)), fma(a.re, b.im, a.im * b.re)};
}
template <class R> __device__ __forceinline__ Cx<R> operator*(R s, Cx<R> a) { return {s * a.re, s * a.im}; }
template <class R> __device__ __forceinline__ Cx<R> operator*(Cx<R> a, R s) { return {s * a.re, s * a.im}; }
template <class R> __device__ __forceinline__ Cx<R> operator/(Cx<R> a, R s) { return {a.re / s, a.im / s}; }
// a * x + y with one rounding per component.  The denoising primal steps
// write div + lambda f with it, so that every kernel rounds it the same way
// (left to the compiler, a kernel that holds f across iterations computed
// lambda f once, rounded, and the one-iteration kernels fused it).
template <class R> __device__ __forceinline__ R fmadd(R a, R x, R y) { return fma(a, x, y); }
template <class R> __device__ __forceinline__ Cx<R> fmadd(R a, Cx<R> x, Cx<R> y) {
  return {fma(a, x.re, y.re), fma(a, x.im, y.im)};
}
// c ? a : b, component-wise (a select, not a branch)
template <class R> __device__ __forceinline__ Cx<R> csel(bool c, Cx<R> a, Cx<R> b) {
  return {c ? a.re : b.re, c ? a.im : b.im};
}
// a * conj(b)
template <class R> __device__ __forceinline__ Cx<R> mulconj(Cx<R> a, Cx<R> b) {
  return {fma(a.re, b.re, a.im * b.im), fma(a.im, b.re, -(a.re * b.im))};
}

template <class P> struct PT { using R = P; static constexpr bool cplx = false; };
template <class R> struct PT<Cx<R>> { using Rt = R; using R_ = R; static constexpr bool cplx = true; };
template <class P> struct RealOf { using T = P; };
template <class R> struct RealOf<Cx<R>> { using T = R; };

template <class P> __device__ __forceinline__ P pzero() { return P(0); }
template <> __device__ __forceinline__ Cx<float> pzero<Cx<float>>() { return {0.f, 0.f}; }
template <> __device__ __forceinline__ Cx<double> pzero<Cx<double>>() { return {0.0, 0.0}; }

__device__ __forceinline__ float abs2(float a) { return a * a; }
__device__ __forceinline__ double abs2(double a) { return a * a; }
template <class R> __device__ __forceinline__ R abs2(Cx<R> a) { return fma(a.re, a.re, a.im * a.im); }  // (as the products above)
// |a|^2 + |b|^2 and |a|^2 + |b|^2 + 2 |c|^2 with explicit fused multiply-adds
// (of two products the compiler fuses either one, and not the same one in
// every kernel).
template <class R> __device__ __forceinline__ R sumsq(R a, R b) { return fma(a, a, b * b); }
template <class R> __device__ __forceinline__ R sumsq(Cx<R> a, Cx<R> b) { return abs2(a) + abs2(b); }
template <class P> __device__ __forceinline__ auto sumsq_sym(P a, P b, P c) { return fma(decltype(abs2(c))(2), abs2(c), sumsq(a, b)); }
__device__ __forceinline__ double dabs2(float a) { return double(a) * double(a); }
__device__ __forceinline__ double dabs2(double a) { return a * a; }
template <class R> __device__ __forceinline__ double dabs2(Cx<R> a) {
  return double(a.re) * double(a.re) + double(a.im) * double(a.im);
}
__device__ __forceinline__ double redot(float a, float b) { return double(a) * double(b); }
__device__ __forceinline__ double redot(double a, double b) { return a * b; }
template <class R> __device__ __forceinline__ double redot(Cx<R> a, Cx<R> b) {
  return double(a.re) * double(b.re) + double(a.im) * double(b.im);
}

// fp16 storage of the TGV duals (compute stays in the pixel type).
template <class P> struct Half;
template <> struct Half<float> { using T = _Float16; };
template <> struct Half<Cx<float>> { using T = Cx<_Float16>; };
template <> struct Half<double> { using T = double; };
template <> struct Half<Cx<double>> { using T = Cx<double>; };

// Device memory reached through the slice descriptors is addressed with
// global-address-space pointers (gptr): loads and stores through them compile
// to global_* instructions with a scalar base, where generic pointers give
// flat_* ones, which also count against the LDS wait counter (so every LDS
// wait of an FFT stage would wait for the outstanding register prefetches).
// (The host pass of the same source, which only checks device code, keeps
// generic pointers.)
#if defined(__HIP_DEVICE_COMPILE__)
template <class T> using G = __attribute__((address_space(1))) T;
template <class T> struct NoAS { using type = T; };
template <class T> struct NoAS<G<T>> { using type = T; };
#else
template <class T> using G = T;
template <class T> struct NoAS { using type = T; };
#endif
template <class T> using Plain = std::remove_const_t<typename NoAS<T>::type>;
template <class T>
__device__ __forceinline__ G<T>* gptr(const void* p) {
  return (G<T>*)(const_cast<void*>(p));
}

// Element access of a plane stored as S (get/put take any pointer to S).
template <class P, class S> struct Ld {
  template <class A> static __device__ __forceinline__ P get(A* a, size_t i) { return a[i]; }
  template <class A> static __device__ __forceinline__ void put(A* a, size_t i, P v) { a[i] = v; }
};
// The value stored is the float result rounded to nearest half: the empty
// register constraint keeps the compiler from fusing the product that
// produced it with the conversion (a mixed-precision FMA rounds once, straight
// to half), so every kernel stores the same halves.
__device__ __forceinline__ _Float16 to_half(float v) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm("" : "+v"(v));
#endif
  return _Float16(v);
}
template <> struct Ld<float, _Float16> {
  template <class A> static __device__ __forceinline__ float get(A* a, size_t i) { return float(a[i]); }
  template <class A> static __device__ __forceinline__ void put(A* a, size_t i, float v) { a[i] = to_half(v); }
};
template <> struct Ld<Cx<float>, Cx<_Float16>> {
  template <class A> static __device__ __forceinline__ Cx<float> get(A* a, size_t i) {
    Cx<_Float16> h = a[i];
    return {float(h.re), float(h.im)};
  }
  template <class A> static __device__ __forceinline__ void put(A* a, size_t i, Cx<float> v) {
    a[i] = Cx<_Float16>{to_half(v.re), to_half(v.im)};
  }
};

// 1 / x: the hardware reciprocal (within 1 ulp) in single precision, a
// correctly rounded division in double precision.
template <class R> __device__ __forceinline__ R rcp(R x) { return R(1) / x; }
template <> __device__ __forceinline__ float rcp<float>(float x) { return __builtin_amdgcn_rcpf(x); }

// The projection onto a ball of radius alpha, as the factor min(1, alpha /
// |b|) from s = |b|^2 and w = ball_weight(alpha).  Single precision: alpha
// times the hardware's reciprocal square root (within 1 ulp), a rounding less
// than sqrt, a product with 1 / alpha and a reciprocal, and 15 instructions
// fewer (the correctly rounded sqrt alone takes about 12).  Double precision:
// correctly rounded steps.  s = 0 gives 1; a negative (-0 too, as max(1, |b| /
// alpha) has it) or NaN alpha projects nothing.
__device__ __forceinline__ float ball_weight(float alpha) {
  return alpha >= 0.f && !__builtin_signbit(alpha) ? alpha : __builtin_inff();
}
__device__ __forceinline__ double ball_weight(double alpha) { return rcp(alpha); }
__device__ __forceinline__ float ball_scale(float s, float w) { return fminf(1.f, w * __builtin_amdgcn_rsqf(s)); }
__device__ __forceinline__ double ball_scale(double s, double w) { return rcp(fmax(1.0, sqrt(s) * w)); }

// The same for any radius: the hardware takes a subnormal s (|b| < 2^-63) for
// zero, hence for inside of every ball, so radii below 2^-63 scale s by 2^24
// first, which makes every s normal (and takes |b| above 2^52 for infinite,
// whose projection is zero).  The product by 1 of the other radii changes no
// bit; it costs the blocked TGV launches 4 % (512 x 512 complex, 1000
// iterations 3.59 against 3.45 ms), which take it for those radii only, and
// the MRI dual steps nothing (320 x 320, 15 coils, 300 iterations 8.36 ms
// against 8.37).
constexpr double kTinyRadius = 0x1p-63;
template <class R> struct Ball {
  R w;
};
template <> struct Ball<float> {
  float w, s;  // weight, scale of |b|^2
};
__device__ __forceinline__ Ball<double> ball_any(double alpha) { return {ball_weight(alpha)}; }
__device__ __forceinline__ Ball<float> ball_any(float alpha) {
  const bool tiny = alpha < float(kTinyRadius);
  return {ball_weight(alpha) * (tiny ? 0x1p12f : 1.f), tiny ? 0x1p24f : 1.f};
}
__device__ __forceinline__ double ball_scale(double s, Ball<double> b) { return ball_scale(s, b.w); }
__device__ __forceinline__ float ball_scale(float s, Ball<float> b) { return ball_scale(s * b.s, b.w); }

// The arithmetic of the dual step at one pixel, on values: c = ubar, uxp /
// uyp = ubar at the forward neighbours (c itself at the last column / row);
// TGV: vx0, vy0 = vbar, vxx = vbar_x and vyx = vbar_y at the x neighbour,
// vxy, vyy at the y neighbour.  Updates p (and q) in place, with optional
// gap terms t[0] += |grad ub - vb|, t[1] += |E vb|_F, t[2] += Re<grad ub -
// vb, p> + Re<E vb, q>_F (TGV_dual_p_kernel / TGV_dual_q_kernel /
// TV_dual_p_kernel).  w0, w1: ball_weight or ball_any of alpha0 (q; TGV only)
// and alpha1 (p; 1 for TV).
template <class P, bool TGV, bool GAP, class B>
__device__ __forceinline__ void dual_math(P c, P uxp, P uyp, P vx0, P vy0, P vxx, P vyx, P vxy, P vyy, P& px, P& py,
                                          P& qxx, P& qyy, P& qxy, typename RealOf<P>::T sigma, B w0, B w1,
                                          double* t) {
  using R = typename RealOf<P>::T;
  P tx = uxp - c, ty = uyp - c;
  if (TGV) {
    tx = tx - vx0;
    ty = ty - vy0;
    const P exx = vxx - vx0;
    const P eyy = vyy - vy0;
    const P exy = R(0.5) * (vxy - vx0 + vyx - vy0);
    const P bxx = qxx + sigma * exx;
    const P byy = qyy + sigma * eyy;
    const P bxy = qxy + sigma * exy;
    const R sq = ball_scale(sumsq_sym(bxx, byy, bxy), w0);
    qxx = bxx * sq;
    qyy = byy * sq;
    qxy = bxy * sq;
    if (GAP) {
      t[1] += sqrt(dabs2(exx) + dabs2(eyy) + 2.0 * dabs2(exy));
      t[2] += redot(exx, qxx) + redot(eyy, qyy) + 2.0 * redot(exy, qxy);
    }
  }
  const P ax = px + sigma * tx;
  const P ay = py + sigma * ty;
  const R sp = ball_scale(sumsq(ax, ay), w1);
  px = ax * sp;
  py = ay * sp;
  if (GAP) {
    t[0] += sqrt(dabs2(tx) + dabs2(ty));
    t[2] += redot(tx, px) + redot(ty, py);
  }
}

__device__ __forceinline__ bool slice_active(const SliceDev& d) { return gptr<const int>(d.ctl)[CTL_ACTIVE] != 0; }

// Workgroups are dispatched round-robin over the 8 XCDs (each with its own
// L2).  Give XCD x a contiguous range of logical work items, so that items
// touching neighbouring memory (adjacent column groups, adjacent rows) share
// one L2.  Bijective on [0, n).
__device__ __forceinline__ int xcd_item(int b, int n) {
  const int q = n >> 3, r = n & 7, x = b & 7, k = b >> 3;
  return x * q + min(x, r) + k;
}

// Workgroup barrier with its own wait for the wave's LDS accesses.  (At the
// head of a loop whose last LDS store is at its end, the compiler drops the
// wait of __syncthreads, which it finds satisfied on the way into the loop:
// read in this build's assembly, where the barrier let a wave read the edge
// row of the iteration before.)
__device__ __forceinline__ void wg_barrier() {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#endif
}

}  // namespace pdt
