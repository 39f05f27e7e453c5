// pdt_block.hip -- temporally blocked denoising: k ROF or TGV iterations per
// launch on tiles held in registers (gfx950).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "pdt_desc.hpp"
#include "pdt_launch.hpp"
#include "pdt_pixel.hpp"

namespace pdt {

namespace {

// The value of the previous / next lane of the wave (0 at its ends).
__device__ __forceinline__ int dpp_prev(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x138, 0xf, 0xf, true); }
__device__ __forceinline__ int dpp_next(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x130, 0xf, 0xf, true); }
__device__ __forceinline__ float lane_prev(float v) { return __builtin_bit_cast(float, dpp_prev(__builtin_bit_cast(int, v))); }
__device__ __forceinline__ float lane_next(float v) { return __builtin_bit_cast(float, dpp_next(__builtin_bit_cast(int, v))); }
__device__ __forceinline__ double lane_prev(double v) { return __hiloint2double(dpp_prev(__double2hiint(v)), dpp_prev(__double2loint(v))); }
__device__ __forceinline__ double lane_next(double v) { return __hiloint2double(dpp_next(__double2hiint(v)), dpp_next(__double2loint(v))); }
template <class R> __device__ __forceinline__ Cx<R> lane_prev(Cx<R> v) { return {lane_prev(v.re), lane_prev(v.im)}; }
template <class R> __device__ __forceinline__ Cx<R> lane_next(Cx<R> v) { return {lane_next(v.re), lane_next(v.im)}; }

__device__ __forceinline__ float sel(bool c, float a, float b) { return c ? a : b; }
__device__ __forceinline__ double sel(bool c, double a, double b) { return c ? a : b; }
template <class R> __device__ __forceinline__ Cx<R> sel(bool c, Cx<R> a, Cx<R> b) { return csel(c, a, b); }

// A value as a store and a load would leave it: the empty register constraint
// keeps the compiler from fusing the product that formed it with its use in
// the next step (the one-iteration kernels, with memory in between, round it).
__device__ __forceinline__ float rounded(float v) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm("" : "+v"(v));
#endif
  return v;
}
__device__ __forceinline__ double rounded(double v) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm("" : "+v"(v));
#endif
  return v;
}
template <class R> __device__ __forceinline__ Cx<R> rounded(Cx<R> v) { return {rounded(v.re), rounded(v.im)}; }

// The value a dual field holds after a store to its storage type S and a
// load back (fp16 storage: rounded to half).
template <class P, class S>
__device__ __forceinline__ P storage_round(P v) {
  if constexpr (std::is_same<P, S>::value) {
    return rounded(v);
  } else {
    S s[1];
    Ld<P, S>::put(s, 0, v);
    return Ld<P, S>::get(s, 0);
  }
}

// Tiles along one axis of n pixels, for regions of `reg` pixels and a halo of
// k: one tile if the region covers the axis (no halo), else interiors of
// reg - 2k, the first and last of up to reg - k (an image border needs no
// halo).
inline int tile_count(int n, int reg, int k) { return n <= reg ? 1 : (n - 2 * k + reg - 2 * k - 1) / (reg - 2 * k); }
__device__ __forceinline__ int tile_lo(int b, int reg, int k) { return b == 0 ? 0 : b * (reg - 2 * k) + k; }
__device__ __forceinline__ int tile_hi(int b, int nb, int n, int reg, int k) { return b == nb - 1 ? n : (b + 1) * (reg - 2 * k) + k; }

// What a launch needs of its slice, by value: the loads of the state wait for
// the kernel arguments only, not for a descriptor in memory or for the launch's
// dimensions, which a kernel reads from memory too.
struct BlockArgs {
  const void *u, *ub, *v, *p, *q, *f;  // the state read
  void *ou, *oub, *ov, *op, *oq;       // and written
  int* ctl;
  int W, H, k, waves, nbx, nby;  // image, iterations, waves of a workgroup, tiles
  double tau, sigma, lambda, theta, alpha0, alpha1;
};

// A point of the program by which the memory accesses before it are issued and
// the launch's parameters and output addresses are in registers.
__device__ __forceinline__ void args_ready(const BlockArgs& d) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" ::"s"(d.ou), "s"(d.ov), "s"(d.op), "s"(d.oq), "s"(d.tau), "s"(d.sigma), "s"(d.lambda), "s"(d.theta),
               "s"(d.alpha0), "s"(d.alpha1)
               : "memory");
#endif
}

// k iterations (TV: TV_dual_p_kernel, TV_primal_u_kernel; TGV, primal step
// first: TV_primal_u_kernel + TGV_primal_v_kernel, TGV_dual_p_kernel +
// TGV_dual_q_kernel; tgv_kernels.cuh:225-324,568-605,647-686,
// tvoptimizer.cu:102-118, tgvoptimizer.cu:119-135) on one tile.
//
// A workgroup's region is 64 columns by NW J rows: wave w holds rows
// [w J, w J + J) in registers, one column per lane.  Of the stencils'
// neighbours, those in y are the lane's own registers, those in x come from
// the next lane (DPP), and only the first and last row of each wave go
// through LDS (what one wave's last row passes to the wave below, edge_dn,
// and its first row to the wave above, edge_up).  The rows that need no
// exchange are computed between the store and the barrier, so the two
// barriers of an iteration are short.  Each iteration the region where the
// values are exact shrinks by one pixel on every side that is not an image
// border (the other values stay finite and are never stored); after k
// iterations the tile's interior is exact and goes to the other copy of the
// state (BlockArgs), so no workgroup reads a halo that another writes.
//
// Image borders: the region's first row and lane are row 0 and column 0 where
// the region touches them (the exchange row above wave 0 and the lane before
// lane 0 read as zero: a backward difference without the subtraction), its
// last row is row H - 1 where it touches that one (the last wave's last row
// has itself as lower neighbour), and column W - 1 is selected per lane.
// Images lower than the region (FLAT) place row H - 1 by selects.
//
// The per-pixel arithmetic is that of k_tv_dual / k_tv_primal and
// k_tgv_primal / k_tgv_dual, in the same order, and duals are rounded to
// their storage type after every dual step, so the iterates equal theirs bit
// for bit.  TGV launches do not store ubar and vbar: the primal step, which
// comes first, rewrites them.
//
// Bound by vector instructions and by what is left of the waits: a launch of 6
// iterations of TGV on 512 x 512 complex pixels takes 19.6 us, of which the
// vector instructions alone 10.4 (2.0 times the image's pixels, with the halo);
// the waves wait 28 % of their time.  TGV with fp16 duals on 961 x 1100: 21.0
// and 13.2 us, 33 %; 20 iterations of TV on 256 x 256: 13.2 and 9.2 us, 36 %.
//
// ANY: projection radii of any size (ball_any).
template <class P, class S, bool TGV, int J, bool FLAT, bool ANY>
__device__ __forceinline__ void block_iterations(const BlockArgs& d, P* smem) {
  using R = typename RealOf<P>::T;
  using L = Ld<P, S>;
  constexpr int NU = TGV ? 3 : 1;  // values a row passes up (ubar, vbar) and down (p_y, q_yy, q_xy)
  const int W = d.W, H = d.H, k = d.k;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  const int NW = d.waves, RH = NW * J;
  const int nbx = d.nbx, nby = d.nby;
  const int b = xcd_item(blockIdx.x, nbx * nby);  // neighbouring tiles on one XCD
  const int by = b / nbx, bx = b - by * nbx;
  const int x0 = tile_lo(bx, kBlockCols, k), x1 = tile_hi(bx, nbx, W, kBlockCols, k);
  const int y0 = tile_lo(by, RH, k), y1 = tile_hi(by, nby, H, RH, k);
  const int xa = max(0, min(bx * (kBlockCols - 2 * k), W - kBlockCols));
  const int ya = FLAT ? 0 : min(by * (RH - 2 * k), H - RH);
  const int x = xa + lane, yw = ya + wave * J;  // this lane's column, its first row
  const size_t n = size_t(W) * H;
  P* const edge_dn = smem;                       // [NW + 1][NU][64], slot 0 zero
  P* const edge_up = smem + (NW + 1) * NU * 64;  // [NW][NU][64]
  int active = 1;
  if constexpr (TGV) active = gptr<const int>(d.ctl)[CTL_ACTIVE];
  P u[J], ub[J], f[J], px[J], py[J], vx[J], vy[J], vbx[J], vby[J], qxx[J], qyy[J], qxy[J];
  {
    const auto gu = gptr<const P>(d.u);
    const auto gb = gptr<const P>(d.ub);
    const auto gv = gptr<const P>(d.v);
    const auto gp = gptr<const S>(d.p);
    const auto gq = gptr<const S>(d.q);
    const auto gf = gptr<const P>(d.f);
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const size_t i = size_t(FLAT ? min(yw + j, H - 1) : yw + j) * W + min(x, W - 1);
      u[j] = gu[i];
      f[j] = gf[i];
      px[j] = L::get(gp, i);
      py[j] = L::get(gp, i + n);
      if constexpr (TGV) {
        vx[j] = gv[i];
        vy[j] = gv[i + n];
        qxx[j] = L::get(gq, i);
        qyy[j] = L::get(gq, i + n);
        qxy[j] = L::get(gq, i + 2 * n);
      } else {
        ub[j] = gb[i];
      }
    }
  }
  // A finished slice's workgroups leave before their first store.  The fence
  // keeps the loads above ahead of this one's wait, where the compiler moved
  // them behind the branch.  ROF reads the control word after its few loads and
  // waits for all of them at once (20 iterations of 256 x 256: 12.9 us, 13.8
  // with the word first, 14.0 without the fence).  TGV reads it first, which
  // keeps its 36 or more loads in flight until their values are stored to LDS,
  // and has the launch's other arguments fetched here, not behind the branch one
  // latency after the other (a launch on 474 x 1065 complex pixels 0.9 %, on 100
  // x 120 1.2 %, on 256 x 300 in double 1.5 % shorter).
  if constexpr (TGV) {
    args_ready(d);
  } else {
    asm volatile("" ::: "memory");
    active = gptr<const int>(d.ctl)[CTL_ACTIVE];
  }
  if (active == 0) return;
  if (wave == 0)
    for (int c = 0; c < NU; ++c) edge_dn[c * 64 + lane] = pzero<P>();
  auto put_dn = [&]() {
    P* e = edge_dn + (wave + 1) * NU * 64 + lane;
    e[0] = py[J - 1];
    if constexpr (TGV) {
      e[64] = qyy[J - 1];
      e[128] = qxy[J - 1];
    }
  };
  auto put_up = [&]() {
    P* e = edge_up + wave * NU * 64 + lane;
    e[0] = ub[0];
    if constexpr (TGV) {
      e[64] = vbx[0];
      e[128] = vby[0];
    }
  };
  const R sigma = R(d.sigma), tau = R(d.tau), lambda = R(d.lambda), theta = R(d.theta);
  auto ball = [](R alpha) {
    if constexpr (ANY) return ball_any(alpha);
    else return ball_weight(alpha);
  };
  const auto w0 = ball(R(TGV ? d.alpha0 : 1.0)), w1 = ball(R(TGV ? d.alpha1 : 1.0));
  const R un_scale = rcp(R(1) + tau * lambda);
  const bool xlast = x >= W - 1, xcut = xlast && W > 1;  // (W = 1: column 0 keeps its value in a backward difference)
  // row H - 1: FLAT by its number, else the last wave's last row.  (Without a
  // lower neighbour that row of any region is inexact after its first dual
  // step; it must not be so after a primal step before it, so the cut of the
  // backward difference is made at the image border only.)
  const bool bottom = (FLAT || ya + RH >= H) && H > 1;
  auto ylast = [&](int j) { return FLAT ? yw + j >= H - 1 : j == J - 1 && wave == NW - 1; };
  auto ycut = [&](int j) { return ylast(j) && bottom; };
  // backward differences: a value without its own part at the last column /
  // row, minus the previous one (zero before the first)
  auto bdx = [&](P c) { return sel(xcut, pzero<P>(), c) - lane_prev(c); };
  auto bdy = [&](int j, P c, P prev) { return sel(ycut(j), pzero<P>(), c) - prev; };
  auto primal = [&](int j, P py_up, P qyy_up, P qxy_up) {
    const P uo = u[j];
    const P div = bdx(px[j]) + bdy(j, py[j], py_up);
    P un = uo + tau * fmadd(lambda, f[j], div);
    un = rounded(un * un_scale);
    u[j] = un;
    ub[j] = (R(1) + theta) * un - theta * uo;
    if constexpr (TGV) {
      const P dsx = bdx(qxx[j]) + bdy(j, qxy[j], qxy_up);
      const P dsy = bdy(j, qyy[j], qyy_up) + bdx(qxy[j]);
      const P ox = vx[j], oy = vy[j];
      const P nx = ox + tau * (dsx + px[j]);
      const P ny = oy + tau * (dsy + py[j]);
      vx[j] = nx;
      vy[j] = ny;
      vbx[j] = (R(1) + theta) * nx - theta * ox;
      vby[j] = (R(1) + theta) * ny - theta * oy;
    }
  };
  auto dual = [&](int j, P ub_dn, P vbx_dn, P vby_dn) {
    auto nx = [&](P c) { return sel(xlast, c, lane_next(c)); };
    auto ny = [&](P c, P next) { return sel(ylast(j), c, next); };
    if constexpr (TGV) {
      dual_math<P, true, false>(ub[j], nx(ub[j]), ny(ub[j], ub_dn), vbx[j], vby[j], nx(vbx[j]), nx(vby[j]),
                                ny(vbx[j], vbx_dn), ny(vby[j], vby_dn), px[j], py[j], qxx[j], qyy[j], qxy[j], sigma, w0,
                                w1, nullptr);
      px[j] = storage_round<P, S>(px[j]);
      py[j] = storage_round<P, S>(py[j]);
      qxx[j] = storage_round<P, S>(qxx[j]);
      qyy[j] = storage_round<P, S>(qyy[j]);
      qxy[j] = storage_round<P, S>(qxy[j]);
    } else {
      const P z = pzero<P>();
      P q0 = z, q1 = z, q2 = z;
      dual_math<P, false, false>(ub[j], nx(ub[j]), ny(ub[j], ub_dn), z, z, z, z, z, z, px[j], py[j], q0, q1, q2, sigma, w0,
                                 w1, nullptr);
      px[j] = rounded(px[j]);
      py[j] = rounded(py[j]);
    }
  };
  // the rows of a half step with their neighbours in this wave, then the one
  // with its neighbour in the next wave
  auto primal_rows = [&]() {
#pragma unroll
    for (int j = 1; j < J; ++j) primal(j, py[j - 1], qyy[j - 1], qxy[j - 1]);
  };
  auto primal_edge = [&]() {
    const P* e = edge_dn + wave * NU * 64 + lane;
    if constexpr (TGV) primal(0, e[0], e[64], e[128]);
    else primal(0, e[0], e[0], e[0]);
  };
  auto dual_rows = [&]() {
#pragma unroll
    for (int j = 0; j < J - 1; ++j) dual(j, ub[j + 1], vbx[j + 1], vby[j + 1]);
  };
  auto dual_edge = [&]() {
    const P* e = edge_up + min(wave + 1, NW - 1) * NU * 64 + lane;  // (the last wave's value is not used)
    if constexpr (TGV) dual(J - 1, e[0], e[64], e[128]);
    else dual(J - 1, e[0], e[0], e[0]);
  };
  if constexpr (TGV) {
    put_dn();
    for (int it = 0; it < k; ++it) {
      primal_rows();
      wg_barrier();
      primal_edge();
      put_up();
      dual_rows();
      wg_barrier();
      dual_edge();
      put_dn();
    }
  } else {
    put_up();
    for (int it = 0; it < k; ++it) {
      dual_rows();
      wg_barrier();
      dual_edge();
      put_dn();
      primal_rows();
      wg_barrier();
      primal_edge();
      put_up();
    }
  }
  const auto ou = gptr<P>(d.ou);
  const auto ob = gptr<P>(d.oub);
  const auto ov = gptr<P>(d.ov);
  const auto op = gptr<S>(d.op);
  const auto oq = gptr<S>(d.oq);
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int y = yw + j;
    if (y >= y0 && y < y1 && x >= x0 && x < x1) {
      const size_t i = size_t(y) * W + x;
      ou[i] = u[j];
      L::put(op, i, px[j]);
      L::put(op, i + n, py[j]);
      if constexpr (TGV) {
        ov[i] = vx[j];
        ov[i + n] = vy[j];
        L::put(oq, i, qxx[j]);
        L::put(oq, i + n, qyy[j]);
        L::put(oq, i + 2 * n, qxy[j]);
      } else {
        ob[i] = ub[j];
      }
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) gptr<int>(d.ctl)[CTL_ITER] += k;
}

template <class P, int J, int NT, bool FLAT>
__global__ __launch_bounds__(NT) void k_tv_block(BlockArgs d) {
  extern __shared__ char smem_raw[];
  block_iterations<P, P, false, J, FLAT, false>(d, reinterpret_cast<P*>(smem_raw));
}
template <class P, class S, int J, int NT, bool FLAT, bool ANY>
__global__ __launch_bounds__(NT) void k_tgv_block(BlockArgs d) {
  extern __shared__ char smem_raw[];
  block_iterations<P, S, true, J, FLAT, ANY>(d, reinterpret_cast<P*>(smem_raw));
}

// Rows per lane and most waves of a workgroup: the state of a pixel is 5 (TV)
// or 12 (TGV) values, in 512 / (waves per SIMD) registers.  Two rows per lane
// measured the same, eight slower (they spill or halve the waves).  Complex
// double TGV spills 19 registers (80 bytes) with four.
template <class P, bool TGV> struct BlockCfg;
template <> struct BlockCfg<float, false> { static constexpr int J = kBlockRows, NW = 16; };
template <> struct BlockCfg<Cx<float>, false> { static constexpr int J = kBlockRows, NW = 16; };
template <> struct BlockCfg<double, false> { static constexpr int J = kBlockRows, NW = 16; };
template <> struct BlockCfg<Cx<double>, false> { static constexpr int J = kBlockRows, NW = 8; };
template <> struct BlockCfg<float, true> { static constexpr int J = kBlockRows, NW = 16; };
template <> struct BlockCfg<Cx<float>, true> { static constexpr int J = kBlockRows, NW = 8; };
template <> struct BlockCfg<double, true> { static constexpr int J = kBlockRows, NW = 8; };
template <> struct BlockCfg<Cx<double>, true> { static constexpr int J = kBlockRows, NW = 8; };

template <class F>
void with_block_cfg(int kind, int dtype, bool fp16, F&& fn) {
  auto go = [&](auto p, auto s) {
    using P = decltype(p);
    using S = decltype(s);
    if (kind == K_TGV) fn(p, s, std::integral_constant<bool, true>{}, BlockCfg<P, true>{});
    else fn(p, p, std::integral_constant<bool, false>{}, BlockCfg<P, false>{});
    (void)sizeof(S);
  };
  switch (dtype) {
    case DT_F32:
      if (fp16 && kind == K_TGV) go(float{}, _Float16{});
      else go(float{}, float{});
      break;
    case DT_C64:
      if (fp16 && kind == K_TGV) go(Cx<float>{}, Cx<_Float16>{});
      else go(Cx<float>{}, Cx<float>{});
      break;
    case DT_F64: go(double{}, double{}); break;
    default: go(Cx<double>{}, Cx<double>{}); break;
  }
}

}  // namespace

BlockShape block_shape(int kind, int dtype, int W, int H, int tx, int ty, int k) {
  BlockShape s;
  if (tx <= 0 || ty <= 0 || k <= 0 || k > 4096) return s;
  with_block_cfg(kind, dtype, false, [&](auto, auto, auto, auto cfg) {
    using B = decltype(cfg);
    // rows of the region: the tile and its halo, whole waves of rows, at most
    // those of NW waves.  Its columns are the 64 lanes of a wave, however
    // narrow the tile: the others would only repeat a neighbour's work (512 x
    // 512 complex TGV, tiles of 32 x 20 pixels and 6 iterations: 5.46 ms per
    // 1000 iterations with 44 lanes in use, 3.46 with 64).
    int waves = (std::min(ty, B::J * B::NW) + 2 * std::min(k, B::J * B::NW) + B::J - 1) / B::J;
    waves = std::min({waves, B::NW, (H + B::J - 1) / B::J});
    const int ry = waves * B::J;
    if ((W > kBlockCols && kBlockCols <= 2 * k) || (H > ry && ry <= 2 * k)) return;  // halo wider than the region
    s.ry = ry;
    s.waves = waves;
    s.nbx = tile_count(W, kBlockCols, k);
    s.grid = s.nbx * tile_count(H, ry, k);
  });
  return s;
}

// The tile by a model of the time of one iteration: a launch costs kLaunchUs
// (its start, the load and store latencies), its bytes (every region loaded,
// the image stored) at kBytesPerUs, and per iteration the rows of the busiest
// CU at the row time of the type, whole waves on each of the 4 SIMDs.  More
// iterations per launch share the first two out over more iterations and
// widen the halo.  Fitted to 1900 measured (type, size, tile) times from 100
// x 120 to 1000 x 1000.  Against the best of 29 tiles, 10 types at 4 sizes: within
// 2 % for 27 of the 40 and 5 % for 35; the worst are at 1000 x 1000, where fewer
// rows per workgroup are faster (complex TGV 11.9 us per iteration and 9.7 with
// 56 x 8 x 4, complex TV 4.28 and 3.62 with 48 x 32 x 8).
void block_choose(int kind, int dtype, bool fp16, int W, int H, int tile[3]) {
  constexpr double kLaunchUs = 4.8, kBytesPerUs = 17e6;
  const bool tgv = kind == K_TGV;
  // us per row of 64 pixels and iteration: float, complex float, double, complex double
  static const double row_us[2][4] = {{0.0077, 0.0168, 0.0256, 0.047}, {0.0273, 0.053, 0.051, 0.082}};
  const double row = row_us[tgv][dtype] * (fp16 ? 1.17 : 1.0);
  const double e = dtype == DT_F32 ? 4 : dtype == DT_C128 ? 16 : 8, pq = fp16 ? e / 2 : e;
  const double load = tgv ? 4 * e + 5 * pq : 5 * e, store = tgv ? 3 * e + 5 * pq : 4 * e;
  double best = 1e300;
  tile[2] = 0;
  for (int k : kBlockIterations)
    for (int waves : kBlockWaves) {
      const int tx = kBlockCols - 2 * k, ty = waves * kBlockRows - 2 * k;
      const BlockShape s = block_shape(kind, dtype, W, H, tx, ty, k);
      if (s.grid == 0 || s.waves < (H < waves * kBlockRows ? 1 : waves)) continue;
      const int per_cu = (s.grid + 255) / 256;
      const double rows = double((per_cu * s.waves + 3) / 4 * 4 * kBlockRows);
      const double bytes = double(s.grid) * s.ry * 64 * load + double(W) * H * store;
      const double us = (kLaunchUs + bytes / kBytesPerUs) / k + rows * row;
      if (us < best) {
        best = us;
        tile[0] = tx;
        tile[1] = ty;
        tile[2] = k;
      }
    }
}

void run_block(const Launch& L, const SliceDev& d, int kind, int dtype, bool fp16, int dir, int k) {
  // (fewer iterations than tb_k: the same region with a larger interior)
  const int more = 2 * (L.tb_k - k);
  const BlockShape s = block_shape(kind, dtype, d.W, d.H, L.tb_x + more, L.tb_y + more, k);
  const BlockArgs a = {dir ? d.u2 : d.u, dir ? d.ub2 : d.ub, dir ? d.v2 : d.v, dir ? d.p2 : d.p, dir ? d.q2 : d.q, d.f,
                       dir ? d.u : d.u2, dir ? d.ub : d.ub2, dir ? d.v : d.v2, dir ? d.p : d.p2, dir ? d.q : d.q2,
                       d.ctl,            d.W,                d.H,              k,                s.waves,
                       s.nbx,            s.grid / s.nbx,     d.tau,            d.sigma,          d.lambda,
                       d.theta,          d.alpha0,           d.alpha1};
  with_block_cfg(kind, dtype, fp16, [&](auto p, auto st, auto tgv, auto cfg) {
    using P = decltype(p);
    using S = decltype(st);
    using B = decltype(cfg);
    constexpr bool TGV = decltype(tgv)::value;
    const size_t lds = size_t(2 * s.waves + 1) * (TGV ? 3 : 1) * 64 * sizeof(P);
    constexpr int J = B::J, NT = 64 * B::NW;
    const dim3 grid(s.grid), block(64 * s.waves);
    auto launch = [&](auto flat, auto any) {
      constexpr bool FLAT = decltype(flat)::value, ANY = decltype(any)::value;
      if constexpr (!TGV) hipLaunchKernelGGL((k_tv_block<P, J, NT, FLAT>), grid, block, lds, L.stream, a);
      else hipLaunchKernelGGL((k_tgv_block<P, S, J, NT, FLAT, ANY>), grid, block, lds, L.stream, a);
    };
    constexpr std::integral_constant<bool, false> no{};
    constexpr std::integral_constant<bool, true> yes{};
    const bool flat = s.ry > d.H;
    if constexpr (TGV && sizeof(typename RealOf<P>::T) == 4) {
      if (std::min(d.alpha0, d.alpha1) < kTinyRadius) return flat ? launch(yes, yes) : launch(no, yes);
    }
    flat ? launch(yes, no) : launch(no, no);
  });
}

}  // namespace pdt
