// Pathwise Greeks of European payoffs by reverse-mode differentiation of the
// Euler scheme (discrete adjoint), one thread per path.
//
// sdepy itself has no Greeks; these kernels differentiate exactly the scheme
// of full_heston_SDE (integration.py:2425-2433, full truncation) and of the
// log-space lognorm/jumpdiff SDEs (integration.py:2127-2130, 2594-2608), on
// the same Philox draws as the forward Euler kernel, so that the price they
// return is the forward kernel's price and the gradients are those of that
// estimator (checked against common-random-number finite differences).
//
// Heston: the variance recursion is not invertible (max(y, 0)), so a reverse
// sweep over the whole path needs its states again.  With an FP64 variance
// the adjoint sweeps segments of a few steps instead, each right after its
// forward steps while their partial derivatives are still in registers, for
// the two adjoint seeds a segment can receive (its final variance and the log
// price), and chains the segments' results forward; nothing is stored or drawn
// twice.  FP32 runs sweep the whole path: pass 1 keeps the variance every C
// steps (checkpoints, C = 8), and the sweep walks the segments backwards,
// recomputing each segment's variances and normals into registers.  In
// segments they would take 2.0 ms in place of 3.15 for 4M x 365, and sum in another
// order, which moves the variance's Greeks by 6e-7: where the variance
// reaches 0, single paths dominate the sums of 1 / sqrt(v).  Which form lies
// nearer to the FP64 values has not been measured.
#include <type_traits>

#include "common.hpp"
#include "philox.hpp"

namespace sdegpu {

// Steps per checkpoint segment of the FP32 adjoint (even: one Philox block
// feeds 2 steps).  8 keeps the segment's registers (3 values per step) small
// enough for 8 waves per SIMD; the checkpoints then cost ~0.7 GB of traffic
// at 4M x 365.
constexpr int kHestonSeg = 8;
// Steps per segment of the FP64 adjoint.  1M x 365: 1.48 ms with 2, 1.47 with
// 4, 1.64 with 8.
constexpr int kHestonSeg64 = 4;
constexpr int kHestonNG = 7;    // x0, r, k, theta, xi, rho, y0
constexpr int kHestonNS = 2 + 2 * kHestonNG;
constexpr int kLogNG = 5;       // x0, mu, sigma, a, b
constexpr int kLogNS = 2 + 2 * kLogNG;

struct HestonArgs {
  const void* steps;  // [n][2] (ds, sqrt ds)
  void* ckpt;         // [nseg][paths] (FP32 adjoint)
  double* part;       // [nblocks][kHestonNS]
  int64_t paths;
  int32_t nsteps, payoff;
  double lx0, x0, r, sig, k, th, xi, rho, rhoc, y0, strike, disc, maturity;
  uint32_t k0, k1, epoch;
};

template <int NS>
__device__ __forceinline__ void block_reduce_store(double (&acc)[NS], double* part) {
  __shared__ double sh[kBlock / 64][NS];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    double v = acc[i];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if (lane == 0) sh[wave][i] = v;
  }
  __syncthreads();
  if (threadIdx.x < NS) {
    double v = 0.0;
#pragma unroll
    for (int w = 0; w < kBlock / 64; ++w) v += sh[w][threadIdx.x];
    part[(int64_t)blockIdx.x * NS + threadIdx.x] = v;
  }
}

template <typename T>
__device__ __forceinline__ T tsqrt(T v);
template <>
__device__ __forceinline__ float tsqrt<float>(float v) {
  return __builtin_amdgcn_sqrtf(v);
}
template <>
__device__ __forceinline__ double tsqrt<double>(double v) {
  return sqrt(v);
}

template <typename T>
__device__ __forceinline__ T trcp(T v);
template <>
__device__ __forceinline__ float trcp<float>(float v) {
  return __builtin_amdgcn_rcpf(v);
}
template <>
__device__ __forceinline__ double trcp<double>(double v) {
  return 1.0 / v;
}

// Per-step constants of the Heston step, built once per launch on the device
// from the caller's (ds, sqrt|ds|) table, in FP64 and then rounded to T:
//   [0] ds            [1] sq = sqrt|ds|   [2] r ds          [3] sigma^2/2 ds
//   [4] k ds          [5] k theta ds      [6] sigma sq zs   [7] xi sq
//   [8] xi sq / 2     [9] sigma sq zs / 2 [10] 1 - k ds
// (zs: the factor the kernels' normals are divided by, kGaussFold)
// With them the forward step is
//   X' = X + (sigma sq sv z0 + (r ds - sigma^2/2 ds y+))
//   V' = V + (xi sq sv w    + (k theta ds - k ds y+)),   w = rho z0 + rhoc z1
// (sv = sqrt(y+), y+ = max(V, 0)), the scheme of full_heston_SDE.sde
// (integration.py:2425-2433).  The kernels add V's increment as one sum and
// X's two state-dependent terms one after the other, with the sum of the
// deterministic r ds added to log x_T after the loop (column 2 is unused
// there); FP64 rounding apart, that is the same scheme.
constexpr int kHestonTab = 12;

// zs multiplies the two columns that meet a normal directly (6 and 9): the
// Greeks kernels draw their FP32 normals divided by zs = kGaussFold<float>.
template <typename T, typename TO = T>
__global__ __launch_bounds__(kBlock) void k_heston_table(const T* __restrict__ steps, int n,
                                                         double r, double sig, double k, double th,
                                                         double xi, double zs, TO* __restrict__ tab,
                                                         double* __restrict__ sum_ds) {
  __shared__ double sh[kBlock];
  double part = 0.0;
  for (int s = threadIdx.x; s < n; s += kBlock) {
    const double ds = (double)steps[2 * s], sq = (double)steps[2 * s + 1];
    TO* row = tab + (int64_t)s * kHestonTab;
    row[0] = (TO)ds;
    row[1] = (TO)sq;
    row[2] = (TO)(r * ds);
    row[3] = (TO)(0.5 * sig * sig * ds);
    row[4] = (TO)(k * ds);
    row[5] = (TO)(k * th * ds);
    row[6] = (TO)(sig * sq * zs);
    row[7] = (TO)(xi * sq);
    row[8] = (TO)(0.5 * xi * sq);
    row[9] = (TO)(0.5 * sig * sq * zs);
    row[10] = (TO)(1.0 - k * ds);
    row[11] = (TO)0;
    part += ds;
  }
  sh[threadIdx.x] = part;
  __syncthreads();
#pragma unroll
  for (int w = kBlock / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) *sum_ds = sh[0];
}

// Derivatives of the full-truncation Heston Euler scheme.
//
// The log-price recursion has unit Jacobian in X, so its adjoint Xbar is the
// payoff's dP/dX_T at every step and every Greek is Xbar times the
// derivative of X_T along a direction.  With
//   a = 1 - k ds + xi sq w / (2 sv),  b = -sigma^2/2 ds + sigma sq z0 / (2 sv)
// where V_n > 0 (d y+/dV = 1), a = 1 and b = 0 elsewhere, a step's partial
// derivatives are dV' = a dV + c, dX' = dX + b dV, with the explicit partials c of
// the directions
//   1: ds               k: theta * 1 - 2,  theta: k * 1
//   2: y+ ds
//   x: sv sq w          xi
//   r: sv sq (z0 - rho w)   rho: times xi / rhoc^2
//   v: none, dV_0 = 1   v0
// (d/d rho of w = rho z0 + rhoc z1 is z0 - rho/rhoc z1 = (z0 - rho w) / rhoc^2).
template <typename T>
__device__ __forceinline__ T pos_part(T v) {
  return v > (T)0 ? v : (T)0;
}
// FP32: one integer max of the bit pattern against 0 (a float max first
// quiets its input, two instructions): a set sign bit is a negative integer,
// so every negative value and -0 give +0 and the rest pass unchanged.
template <>
__device__ __forceinline__ float pos_part<float>(float v) {
  const int b = __builtin_bit_cast(int, v);
  return __builtin_bit_cast(float, b > 0 ? b : 0);
}

// Waves per SIMD the Heston kernels are built for: FP32 8, FP32 with an FP64
// variance state 4 (its variance registers take twice the room), FP64 1.
template <typename T, typename TV>
constexpr int heston_waves() {
  return sizeof(TV) == 8 ? (sizeof(T) == 4 ? 4 : 1) : 8;
}

// One path's state and the derivatives of (X, V) along the five directions.
// The log price is held in T, the variance and every derivative in TV (T, or
// FP64 with FP32 normals).  The normals are those of normals4_folded
// (divided by kGaussFold<T>): rho and rhoc come multiplied by it, table
// columns 6 and 9 too, and the rho direction is taken per unit of it
// (rho_r = rho / kGaussFold<T>).
template <typename T, typename TV>
struct HestonPath {
  T X;
  TV V;
  TV x1, v1, x2, v2, xx, vx, xr, vr, xv, vv;
};

// The partial derivatives of one step (the direction-1 partial is the
// table's ds).
template <typename TV>
struct HestonPartials {
  TV a, b, c2, cx, cr;
};

// Steps (X, V) by the table row at rx, r with the normals z0, z1; the partials
// there.  FLAT forms both selected partials on every lane; otherwise the
// compiler puts each behind a branch with its own scalar loads and a wait for
// them.  1M x 365 FP64: adjoint 1.48 ms flat, 1.52 with the branches; tangent
// 1.53 flat, 1.50 with the branches (FP32, 4M x 365: 2.04 and 1.92).
template <bool FLAT, typename T, typename TV>
__device__ __forceinline__ HestonPartials<TV> heston_step(HestonPath<T, TV>& p,
                                                          const T* __restrict__ rx,
                                                          const TV* __restrict__ r, T z0t, T z1t,
                                                          TV rho, TV rhoc, TV rho_r) {
  HestonPartials<TV> d;
  const TV z0 = (TV)z0t;
  const TV w = rho * z0 + rhoc * (TV)z1t;
  const TV vp = pos_part(p.V);
  const TV sv = tsqrt<TV>(vp);
  const TV h = trcp<TV>(sv);
  const bool pos = sv > (TV)0;
  if constexpr (FLAT) {
    TV da = fma(w * r[8], h, r[10]), db = fma(z0 * r[9], h, -r[3]);
    asm("" : "+v"(da), "+v"(db));
    d.a = pos ? da : (TV)1;
    d.b = pos ? db : (TV)0;
  } else {
    d.a = pos ? fma(w * r[8], h, r[10]) : (TV)1;
    d.b = pos ? fma(z0 * r[9], h, -r[3]) : (TV)0;
  }
  const TV ssq = sv * r[1];
  d.c2 = vp * r[0];
  d.cx = ssq * w;
  d.cr = ssq * fma(-rho_r, w, z0);
  // the deterministic r ds terms are added once, after the loop
  p.X = fma(-rx[3], (T)vp, fma((T)sv * rx[6], z0t, p.X));
  p.V = p.V + fma(-r[4], vp, fma(sv * r[7], w, r[5]));
  return d;
}

// Carries the derivatives over one step (forward mode).
template <typename T, typename TV>
__device__ __forceinline__ void heston_tangent_step(HestonPath<T, TV>& p,
                                                    const HestonPartials<TV>& d, TV ds) {
  p.x1 = fma(p.v1, d.b, p.x1);
  p.v1 = fma(p.v1, d.a, ds);
  p.x2 = fma(p.v2, d.b, p.x2);
  p.v2 = fma(p.v2, d.a, d.c2);
  p.xx = fma(p.vx, d.b, p.xx);
  p.vx = fma(p.vx, d.a, d.cx);
  p.xr = fma(p.vr, d.b, p.xr);
  p.vr = fma(p.vr, d.a, d.cr);
  p.xv = fma(p.vv, d.b, p.xv);
  p.vv = p.vv * d.a;
}

template <typename T, typename TV>
__device__ __forceinline__ HestonPath<T, TV> heston_start(const HestonArgs& a) {
  HestonPath<T, TV> p = {};
  p.X = (T)a.lx0;
  p.V = (TV)a.y0;
  p.vv = (TV)1;
  return p;
}

// Payoff, Greeks and their squares of one path.
template <typename T, typename TV>
__device__ __forceinline__ void heston_greeks_of(const HestonArgs& a, const HestonPath<T, TV>& p,
                                                 double sum_ds, double (&acc)[kHestonNS]) {
  const double S = exp((double)p.X + a.r * sum_ds);
  const bool call = a.payoff == 0;
  const double intr = call ? S - a.strike : a.strike - S;
  const bool itm = intr > 0.0;
  const double pay = itm ? a.disc * intr : 0.0;
  // dP/dX_T = disc * (+-S) on the money
  const double xbar = itm ? (call ? a.disc * S : -a.disc * S) : 0.0;
  const double d1 = (double)p.x1;
  // out of the money every Greek is 0, whatever the derivatives hold
  const double g[kHestonNG] = {
      xbar / a.x0,
      xbar * sum_ds - a.maturity * pay,
      itm ? xbar * (a.th * d1 - (double)p.x2) : 0.0,
      itm ? xbar * a.k * d1 : 0.0,
      itm ? xbar * (double)p.xx : 0.0,
      itm ? xbar * a.xi / (a.rhoc * a.rhoc) * kGaussFold<T> * (double)p.xr : 0.0,
      itm ? xbar * (double)p.xv : 0.0};
  acc[0] = pay;
  acc[1] = pay * pay;
#pragma unroll
  for (int i = 0; i < kHestonNG; ++i) {
    acc[2 + 2 * i] = g[i];
    acc[3 + 2 * i] = g[i] * g[i];
  }
}

// Running reverse-sweep state of one path: the variance adjoint and the four
// parameter sums, all per unit of the constant log-price adjoint Xbar (every
// term of the variance adjoint is Xbar times a path quantity, so the sweep
// carries U = Vbar / Xbar and the sums are scaled by Xbar once at the end).
struct HestonRev {
  float vbar, s1, s2, sx, sr;
};

// One checkpoint segment of the reverse sweep: recompute the segment's
// variances and normals from its checkpoint and the Philox counters into
// registers, then walk its steps backwards.  FULL segments hold C steps.
// rho, rhoc and rho_r as in heston_step.
template <int C, bool FULL, bool KEY1ST>
__device__ __forceinline__ void heston_segment(const HestonArgs& a, const float* __restrict__ tb,
                                               const float* __restrict__ ck, int64_t gid,
                                               uint32_t path, int c, int n, float rho, float rhoc,
                                               float rho_r, HestonRev& rv) {
  const int s0 = c * C;
  float svs[C], ws[C], z0s[C];
  float v = ck[(int64_t)c * a.paths + gid];
#pragma unroll
  for (int j = 0; j < C; j += 2) {
    if (FULL || s0 + j < n) {
      __asm__ volatile("" ::: "memory");
      float z[4];
      normals4_folded<float, KEY1ST>((uint32_t)((s0 + j) >> 1), path, kStreamNormal, a.epoch,
                                     a.k0, a.k1, z);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int s = s0 + j + q;
        z0s[j + q] = z[2 * q];
        ws[j + q] = rho * z[2 * q] + rhoc * z[2 * q + 1];
        if (FULL || s < n) {
          const float* r = tb + (int64_t)s * kHestonTab;
          const float vp = pos_part(v);
          const float sv = tsqrt<float>(vp);
          svs[j + q] = sv;
          v = v + fma(-r[4], vp, fma(sv * r[7], ws[j + q], r[5]));
        }
      }
    }
  }
#pragma unroll
  for (int j = C - 1; j >= 0; --j) {
    const int s = s0 + j;
    if (FULL || s < n) {
      // keep the scalar table loads next to their step: hoisting all of a
      // segment's rows at once overflows the SGPR file into VGPR lanes
      __asm__ volatile("" ::: "memory");
      const float* r = tb + (int64_t)s * kHestonTab;
      const float sv = svs[j], z0 = z0s[j], w = ws[j];
      const float vb = rv.vbar;
      const float u = vb * r[0];
      rv.s1 = rv.s1 + u;
      rv.s2 = fma(u, sv * sv, rv.s2);
      const float b = vb * (sv * r[1]);
      rv.sx = fma(b, w, rv.sx);
      rv.sr = fma(b, fma(-rho_r, w, z0), rv.sr);
      const float h = trcp<float>(sv);
      const float c1 = fma(w, h * r[8], -r[4]);
      const float c2 = fma(z0, h * r[9], -r[3]);
      const float d = fma(vb, c1, c2);
      rv.vbar = sv > 0.f ? vb + d : vb;
    }
  }
}

// Reverse mode over the whole path in FP32, from variance checkpoints.  The
// adjoint of V carries U = Vbar / Xbar; k and theta need the sums of U ds and
// U y+ ds, xi and rho those of U sv sq w and U sv sq (z0 - rho w): the
// derivatives of X_T along the same directions.
template <int C, bool KEY1ST>
__global__ __launch_bounds__(kBlock, (heston_waves<float, float>())) void k_heston_adjoint(
    const HestonArgs a, const float* __restrict__ tb, float* __restrict__ ck,
    const double* __restrict__ sum_ds) {
  static_assert(C % 2 == 0, "one Philox block feeds two steps");
  const int64_t gid = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  const bool live = gid < a.paths;
  const uint32_t path = (uint32_t)gid;
  const int64_t P = a.paths;
  const int n = a.nsteps;
  constexpr double zf = kGaussFold<float>;
  const float rho = (float)(a.rho * zf), rhoc = (float)(a.rhoc * zf), rho_r = (float)(a.rho / zf);

  double acc[kHestonNS];
#pragma unroll
  for (int i = 0; i < kHestonNS; ++i) acc[i] = 0.0;

  if (live) {
    HestonPath<float, float> p = heston_start<float, float>(a);
    // ---- pass 1: forward, variance checkpoints every C steps ----
    for (int s0 = 0; s0 < n; s0 += 2) {
      float z[4];
      normals4_folded<float, KEY1ST>((uint32_t)(s0 >> 1), path, kStreamNormal, a.epoch, a.k0,
                                     a.k1, z);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int s = s0 + j;
        if (s < n) {
          if (s % C == 0) ck[(int64_t)(s / C) * P + gid] = p.V;
          const float* r = tb + (int64_t)s * kHestonTab;
          const float z0 = z[2 * j];
          const float w = rho * z0 + rhoc * z[2 * j + 1];
          const float vp = pos_part(p.V);
          const float sv = tsqrt<float>(vp);
          // the deterministic r ds terms are added once, after the loop
          p.X = fma(-r[3], vp, fma(sv * r[6], z0, p.X));
          p.V = p.V + fma(-r[4], vp, fma(sv * r[7], w, r[5]));
        }
      }
    }
    // ---- reverse sweep over the checkpoint segments, per unit of Xbar ----
    // Full segments run without step guards; only the last one can be short.
    HestonRev rv{0.f, 0.f, 0.f, 0.f, 0.f};
    const int nfull = n / C;
    if (nfull * C < n)
      heston_segment<C, false, KEY1ST>(a, tb, ck, gid, path, nfull, n, rho, rhoc, rho_r, rv);
    for (int c = nfull - 1; c >= 0; --c)
      heston_segment<C, true, KEY1ST>(a, tb, ck, gid, path, c, n, rho, rhoc, rho_r, rv);
    p.x1 = rv.s1;
    p.x2 = rv.s2;
    p.xx = rv.sx;
    p.xr = rv.sr;
    p.xv = rv.vbar;
    heston_greeks_of(a, p, *sum_ds, acc);
  }
  block_reduce_store<kHestonNS>(acc, a.part);
}

// Reverse mode segment by segment (FP64 variance).  After the C forward steps of a segment
// its partials are in registers, and two adjoints are swept back over them
// together: lam, of the segment's final variance (seed 1), and mu, of the
// log price (seed 1; its own recursion is the identity).  Per step, with the
// partials c of each direction,
//   dX += mu c,  G += lam c,  mu <- a mu + b,  lam <- a lam,
// so that at the segment's start d X_end/d V_start = mu, d V_end/d V_start =
// lam and G holds d V_end along the directions; the segments are then chained
// by dX += mu dV, dV <- lam dV + G.  The last step's sweep is free (lam = 1,
// mu = 0), which pays for the chaining: 10 FMAs per step.
//
// VALU-bound (the Philox draws and Box-Muller are half of the
// instructions).  The reverse sweep over the whole path drew every normal
// twice and moved the variance checkpoints: 1M x 365 FP64 2.50 ms with it,
// 1.47 ms now; FP32 with an FP64 variance 1.67 and 1.07 ms.
// tb: the step constants in T (the log-price update); tv: the same in TV
// (tv == tb when TV == T).
template <typename T, typename TV, int C>
__global__ __launch_bounds__(kBlock, (heston_waves<T, TV>())) void k_heston_adjoint_seg(
    const HestonArgs a, const T* __restrict__ tb, const TV* __restrict__ tv,
    const double* __restrict__ sum_ds) {
  static_assert(C % 2 == 0, "one Philox block feeds two steps");
  gauss_init<T>();
  const int64_t gid = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  const bool live = gid < a.paths;
  const uint32_t path = (uint32_t)gid;
  const int n = a.nsteps;
  constexpr double zf = kGaussFold<T>;
  const TV rho = (TV)(a.rho * zf), rhoc = (TV)(a.rhoc * zf), rho_r = (TV)(a.rho / zf);

  double acc[kHestonNS];
#pragma unroll
  for (int i = 0; i < kHestonNS; ++i) acc[i] = 0.0;

  if (live) {
    HestonPath<T, TV> p = heston_start<T, TV>(a);
    int s0 = 0;
    for (; s0 + C <= n; s0 += C) {
      HestonPartials<TV> d[C];
#pragma unroll
      for (int j = 0; j < C; j += 2) {
        T z[4];
        normals4_folded<T>((uint32_t)((s0 + j) >> 1), path, kStreamNormal, a.epoch, a.k0, a.k1,
                           z);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int64_t row = (int64_t)(s0 + j + q) * kHestonTab;
          d[j + q] = heston_step<true, T, TV>(p, tb + row, tv + row, z[2 * q], z[2 * q + 1], rho, rhoc,
                                        rho_r);
        }
      }
      const TV* r = tv + (int64_t)(s0 + C - 1) * kHestonTab;
      TV g1 = r[0], g2 = d[C - 1].c2, gx = d[C - 1].cx, gr = d[C - 1].cr;
      TV lam = d[C - 1].a, mu = d[C - 1].b;
#pragma unroll
      for (int j = C - 2; j >= 0; --j) {
        r -= kHestonTab;
        p.x1 = fma(mu, r[0], p.x1);
        g1 = fma(lam, r[0], g1);
        p.x2 = fma(mu, d[j].c2, p.x2);
        g2 = fma(lam, d[j].c2, g2);
        p.xx = fma(mu, d[j].cx, p.xx);
        gx = fma(lam, d[j].cx, gx);
        p.xr = fma(mu, d[j].cr, p.xr);
        gr = fma(lam, d[j].cr, gr);
        mu = fma(mu, d[j].a, d[j].b);
        lam = lam * d[j].a;
      }
      p.x1 = fma(mu, p.v1, p.x1);
      p.v1 = fma(lam, p.v1, g1);
      p.x2 = fma(mu, p.v2, p.x2);
      p.v2 = fma(lam, p.v2, g2);
      p.xx = fma(mu, p.vx, p.xx);
      p.vx = fma(lam, p.vx, gx);
      p.xr = fma(mu, p.vr, p.xr);
      p.vr = fma(lam, p.vr, gr);
      p.xv = fma(mu, p.vv, p.xv);
      p.vv = lam * p.vv;
    }
    // the steps past the last whole segment, one at a time
    for (; s0 < n; s0 += 2) {
      T z[4];
      normals4_folded<T>((uint32_t)(s0 >> 1), path, kStreamNormal, a.epoch, a.k0, a.k1, z);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        if (s0 + q < n) {
          const int64_t row = (int64_t)(s0 + q) * kHestonTab;
          const HestonPartials<TV> d = heston_step<true, T, TV>(p, tb + row, tv + row, z[2 * q],
                                                          z[2 * q + 1], rho, rhoc, rho_r);
          heston_tangent_step(p, d, tv[row]);
        }
      }
    }
    heston_greeks_of(a, p, *sum_ds, acc);
  }
  block_reduce_store<kHestonNS>(acc, a.part);
}

// Forward mode (tangent): the derivatives are carried along step by step.
template <typename T, typename TV>
__global__ __launch_bounds__(kBlock, (heston_waves<T, TV>())) void k_heston_tangent(
    const HestonArgs a, const T* __restrict__ tb, const TV* __restrict__ tv,
    const double* __restrict__ sum_ds) {
  gauss_init<T>();
  const int64_t gid = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  const bool live = gid < a.paths;
  const uint32_t path = (uint32_t)gid;
  const int n = a.nsteps;
  constexpr double zf = kGaussFold<T>;
  const TV rho = (TV)(a.rho * zf), rhoc = (TV)(a.rhoc * zf), rho_r = (TV)(a.rho / zf);

  double acc[kHestonNS];
#pragma unroll
  for (int i = 0; i < kHestonNS; ++i) acc[i] = 0.0;

  if (live) {
    HestonPath<T, TV> p = heston_start<T, TV>(a);
    auto pair = [&](int s0, int most) {
      T z[4];
      normals4_folded<T>((uint32_t)(s0 >> 1), path, kStreamNormal, a.epoch, a.k0, a.k1, z);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if (j < most) {
          const int64_t row = (int64_t)(s0 + j) * kHestonTab;
          const HestonPartials<TV> d = heston_step<false, T, TV>(p, tb + row, tv + row, z[2 * j],
                                                          z[2 * j + 1], rho, rhoc, rho_r);
          heston_tangent_step(p, d, tv[row]);
        }
      }
    };
    int s0 = 0;
    for (; s0 + 2 <= n; s0 += 2) pair(s0, 2);
    if (s0 < n) pair(s0, 1);
    heston_greeks_of(a, p, *sum_ds, acc);
  }
  block_reduce_store<kHestonNS>(acc, a.part);
}

// ---- lognormal / Merton jump-diffusion (log-space, linear recursion) ----
//
// log x_T = log x0 + sum (mu - sigma^2/2) ds + sigma sum dw + sum_jumps (a + b z):
// the recursion is linear with state-independent coefficients, so its
// adjoint is constant along the path (xbar_n = xbar_T) and the parameter
// adjoints reduce to sums collected in the forward pass.

struct LogArgs {
  const void* steps;        // [n][2] (ds, sqrt ds)
  const double* pois;       // [n][3] (lam ds, exp(-lam ds), zero-count bound) or null
  double* part;             // [nblocks][kLogNS]
  int64_t paths;
  int32_t nsteps, payoff;
  double lx0, x0, mu, sig, ja, jb, strike, disc, maturity;
  uint32_t kw0, kw1, ew, kj0, kj1, ej;
};

constexpr int kLogEvents = 4;  // jump steps per path whose sizes are drawn after the loop

template <typename T>
__global__ __launch_bounds__(kBlock) void k_loglin_greeks(const LogArgs a,
                                                          const T* __restrict__ st,
                                                          const double* __restrict__ pois) {
  gauss_init<T>();
  const int64_t gid = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  const bool live = gid < a.paths;
  const uint32_t path = (uint32_t)gid;
  const int n = a.nsteps;
  const T ja = (T)a.ja, jb = (T)a.jb;
  double acc[kLogNS];
#pragma unroll
  for (int i = 0; i < kLogNS; ++i) acc[i] = 0.0;
  if (live) {
    // log x_T = log x0 + (mu - sigma^2/2) T + sigma sum dw + sum dj: only
    // the sums of dw (which the sigma Greek needs anyway) and of the jump
    // sizes are carried through the steps, and log x_T is formed once in FP64
    T sdw = (T)0, szeta = (T)0, sj = (T)0;
    int njump = 0;
    // Sum of the cnt jump sizes of step s and of their normals: the jump
    // normals of (step s, jump q) are lane q % 4 of block (s, path,
    // jump stream | (q / 4) << 8), as in the Euler kernel.
    auto jumps = [&](int s, int cnt, T& dj, T& zsum) {
      T zz[4];
      for (int q = 0; q < cnt; ++q) {
        if ((q & 3) == 0)
          normals4<T>((uint32_t)s, path, kStreamJump | ((uint32_t)(q >> 2) << 8), a.ej, a.kj0,
                      a.kj1, zz);
        const int l = q & 3;
        const T zq = l == 0 ? zz[0] : l == 1 ? zz[1] : l == 2 ? zz[2] : zz[3];
        dj = dj + (ja + jb * zq);
        zsum = zsum + zq;
      }
    };
    // The log-space recursion is linear with state-independent
    // coefficients and only x_T is needed, so the jump sizes can be added
    // after the step loop: up to kLogEvents jump steps per path are recorded
    // and drawn afterwards, when every lane of the wave draws its own (at lambda
    // ds = 1/252 a wave otherwise draws a Philox block at about one step in five
    // for a single jumping lane).  Further jump steps, counts above 255 and
    // steps beyond 2^24 are drawn in place.  An event is (s << 8 | count); in FP32
    // the step and its Poisson word, which is inverted afterwards too (2M x
    // 252 514 -> 489 us; FP64 was 3% slower so): a bound of 1 or more means
    // a lambda ds below 22.2, whose counts never come near 256.
    // the events live in LDS, one column per lane: recording one is a store
    // at a lane-computed address, not a select into each register
    constexpr bool kLate = sizeof(T) == 4;
    using Event = std::conditional_t<kLate, uint2, uint32_t>;
    __shared__ Event ev[kLogEvents][kBlock];
    int nev = 0;
    auto count = [&](int s, uint32_t word) {
      return poisson_inv(u01_f64(word), pois[3 * s], pois[3 * s + 1], 4096);
    };
    // four steps; groups that are whole run without a test for the last step
    auto group = [&](int s0, auto whole) {
      T z[4];
      normals4<T>((uint32_t)(s0 >> 2), path, kStreamNormal, a.ew, a.kw0, a.kw1, z);
      uint32_t up[4] = {0u, 0u, 0u, 0u};
      if (a.pois) {
        const ctr4 r = philox4x32_10(ctr4{(uint32_t)(s0 >> 2), path, kStreamPoisson, a.ej}, a.kj0, a.kj1);
        up[0] = r.x;
        up[1] = r.y;
        up[2] = r.z;
        up[3] = r.w;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int s = s0 + j;
        if (decltype(whole)::value || s < n) {
          const T dw = z[j] * st[2 * s + 1];
          // a word below the step's bound (the low word of pois[s][2]) is a
          // count of 0: one integer compare in place of forming the FP64
          // uniform; words at or above it take the inversion, which
          // re-checks against exp(-lam ds)
          if (a.pois && up[j] >= reinterpret_cast<const uint32_t*>(pois)[6 * s + 4]) {
            bool kept = false;
            if constexpr (kLate) {
              if (reinterpret_cast<const uint32_t*>(pois)[6 * s + 4] > 0u && nev < kLogEvents &&
                  s < (1 << 24)) {
                ev[nev][threadIdx.x] = make_uint2((uint32_t)s, up[j]);
                ++nev;
                kept = true;
              }
            }
            const int cnt = kept ? 0 : count(s, up[j]);
            if (cnt > 0) {
              if (nev < kLogEvents && cnt < 256 && s < (1 << 24)) {
                if constexpr (kLate) {
                  ev[nev][threadIdx.x] = make_uint2((uint32_t)s, up[j]);
                } else {
                  njump += cnt;
                  ev[nev][threadIdx.x] = ((uint32_t)s << 8) | (uint32_t)cnt;
                }
                ++nev;
              } else {
                njump += cnt;
                T dj = (T)0, zsum = (T)0;
                jumps(s, cnt, dj, zsum);
                sj = sj + dj;
                szeta = szeta + zsum;
              }
            }
          }
          sdw = sdw + dw;
        }
      }
    };
    int s0 = 0;
    for (; s0 + 4 <= n; s0 += 4) group(s0, std::true_type{});
    if (s0 < n) group(s0, std::false_type{});
#pragma unroll
    for (int k = 0; k < kLogEvents; ++k) {
      if (k < nev) {
        T dj = (T)0, zsum = (T)0;
        const Event e = ev[k][threadIdx.x];
        if constexpr (kLate) {
          const int cnt = count((int)e.x, e.y);
          njump += cnt;
          jumps((int)e.x, cnt, dj, zsum);
        } else {
          jumps((int)(e >> 8), (int)(e & 255u), dj, zsum);
        }
        sj = sj + dj;
        szeta = szeta + zsum;
      }
    }
    const double X = a.lx0 + (a.mu - a.sig * a.sig / 2) * a.maturity + a.sig * (double)sdw +
                     (double)sj;
    const double S = exp(X);
    const bool call = a.payoff == 0;
    const double intr = call ? S - a.strike : a.strike - S;
    const bool itm = intr > 0.0;
    const double pay = itm ? a.disc * intr : 0.0;
    const double xbar = itm ? (call ? a.disc * S : -a.disc * S) : 0.0;
    const double g[kLogNG] = {xbar / a.x0, xbar * a.maturity,
                              xbar * (-a.sig * a.maturity + (double)sdw),
                              xbar * (double)njump, xbar * (double)szeta};
    acc[0] = pay;
    acc[1] = pay * pay;
#pragma unroll
    for (int i = 0; i < kLogNG; ++i) {
      acc[2 + 2 * i] = g[i];
      acc[3 + 2 * i] = g[i] * g[i];
    }
  }
  block_reduce_store<kLogNS>(acc, a.part);
}

// The columns' sums of part[rows][ncol], in a fixed order that does not depend on
// scheduling.  Above kSumRows rows the rows are first summed in place, slice by
// slice: a block per slice reads its rows in whole lines and leaves their sum in
// the first.  One block per column reads 8 bytes of every line of all rows, 27
// us for the 15,625 rows of 4M paths, however many loads are in flight; the
// two kernels take 15.  For the 7,813 rows of 2M paths it is 12 and 10, for 1,172 the second
// launch costs 2 more than it saves.
constexpr int kSumRows = 4096, kSumSlices = 64;

__global__ __launch_bounds__(kBlock) void k_sum_slices(double* __restrict__ part, int64_t rows,
                                                       int ncol, int64_t per) {
  __shared__ double sh[kBlock];
  const int64_t lo = blockIdx.x * per, hi = lo + per < rows ? lo + per : rows;
  const int deep = kBlock / ncol;  // rows read at a time
  const int t = threadIdx.x, c = t % ncol, r = t / ncol;
  double v = 0.0;
  if (r < deep)
    for (int64_t i = lo + r; i < hi; i += deep) v += part[i * ncol + c];
  sh[t] = v;
  __syncthreads();
  if (t < ncol) {
    double s = 0.0;
    for (int k = 0; k < deep; ++k) s += sh[k * ncol + t];
    part[lo * ncol + t] = s;
  }
}

// out[c]: the sum of part[r step][c], r < rows, one block per column; each thread
// keeps 4 loads in flight
constexpr int kSumThreads = 1024;

__global__ __launch_bounds__(kSumThreads) void k_sum_columns(const double* __restrict__ part,
                                                             int64_t rows, int64_t step, int ncol,
                                                             double* __restrict__ out) {
  constexpr int kAhead = kSumRows / kSumThreads;
  __shared__ double sh[kSumThreads / 64];
  double v = 0.0;
  for (int64_t r0 = threadIdx.x; r0 < rows; r0 += kAhead * kSumThreads) {
    double q[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int64_t r = r0 + i * kSumThreads;
      q[i] = r < rows ? part[r * step * ncol + blockIdx.x] : 0.0;
    }
#pragma unroll
    for (int i = 0; i < kAhead; ++i) v += q[i];
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kSumThreads / 64; ++w) s += sh[w];
    out[blockIdx.x] = s;
  }
}

static int sum_columns(double* part, int64_t rows, int ncol, double* out, hipStream_t st) {
  int64_t step = 1;
  if (rows > kSumRows) {
    step = (rows + kSumSlices - 1) / kSumSlices;
    const int64_t slices = (rows + step - 1) / step;
    hipLaunchKernelGGL(k_sum_slices, dim3((unsigned)slices), dim3(kBlock), 0, st, part, rows, ncol,
                       step);
    if (int e = launch_status("k_sum_slices")) return e;
    rows = slices;
  }
  hipLaunchKernelGGL(k_sum_columns, dim3(ncol), dim3(kSumThreads), 0, st, (const double*)part, rows, step,
                     ncol, out);
  return launch_status("k_sum_columns");
}

// Workspace of one Heston Greeks launch, in this order (each part 256-byte
// aligned): the per-step table [n][kHestonTab] of the dtype, with an FP64
// variance state the same table in FP64, the FP64 sum of ds, for an FP32
// adjoint the variance checkpoints [nseg][paths], and the per-block partial
// sums.
struct HestonWs {
  size_t tab, tabv, sum, ckpt, part, total;
};

static size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

static HestonWs heston_ws(int dtype, bool v64, int method, int64_t paths, int nsteps) {
  const size_t es = dtype == SDEGPU_F32 ? 4 : 8;
  const size_t ev = v64 ? 8 : es;
  const size_t rows = (size_t)(nsteps > 0 ? nsteps : 1) * kHestonTab;
  HestonWs w;
  w.tab = 0;
  w.tabv = align256(rows * es);
  w.sum = w.tabv + (ev != es ? align256(rows * ev) : 0);
  const int64_t nseg = ev == 4 && method == 0 ? (nsteps + kHestonSeg - 1) / kHestonSeg : 0;
  w.ckpt = w.sum + 256;
  w.part = w.ckpt + align256((size_t)nseg * (size_t)paths * ev);
  w.total = w.part + (size_t)blocks_for(paths) * kHestonNS * sizeof(double);
  return w;
}

}  // namespace sdegpu

using namespace sdegpu;

extern "C" size_t sdegpu_heston_greeks_workspace(const sdegpu_heston_greeks* g) {
  if (!g || g->paths < 1) return 0;
  // (method 0's, which is the larger: one workspace serves both methods)
  return heston_ws(g->dtype, g->variance_f64 != 0, 0, g->paths, g->nsteps).total;
}

extern "C" int sdegpu_heston_greeks_run(const sdegpu_heston_greeks* g, double* out, void* ws,
                                        size_t ws_bytes, void* stream) {
  if (!g || !out) return fail(SDEGPU_EINVAL, "heston_greeks: null argument");
  if (g->dtype != SDEGPU_F32 && g->dtype != SDEGPU_F64)
    return fail(SDEGPU_EUNSUPPORTED, "heston_greeks: dtype code %d", g->dtype);
  if (g->paths < 1 || g->paths > kMaxPaths || g->nsteps < 1)
    return fail(SDEGPU_EINVAL, "heston_greeks: paths=%lld steps=%d", (long long)g->paths,
                g->nsteps);
  if (!g->steps) return fail(SDEGPU_EINVAL, "heston_greeks: missing step table");
  if (!(g->x0 > 0.0) || !(g->rho > -1.0 && g->rho < 1.0))
    return fail(SDEGPU_EINVAL, "heston_greeks: need x0 > 0 and |rho| < 1");
  if (g->payoff != 0 && g->payoff != 1)
    return fail(SDEGPU_EINVAL, "heston_greeks: payoff kind %d", g->payoff);
  if (g->method != 0 && g->method != 1)
    return fail(SDEGPU_EINVAL, "heston_greeks: method %d", g->method);
  if (g->variance_f64 != 0 && g->variance_f64 != 1)
    return fail(SDEGPU_EINVAL, "heston_greeks: variance_f64 %d", g->variance_f64);
  // an FP64 variance state with FP32 normals (FP64 runs carry it anyway)
  const bool v64 = g->variance_f64 != 0 && g->dtype == SDEGPU_F32;
  const HestonWs lay = heston_ws(g->dtype, v64, g->method, g->paths, g->nsteps);
  if (!ws || ws_bytes < lay.total)
    return fail(SDEGPU_ENOMEM, "heston_greeks: workspace of %zu bytes, %zu needed", ws_bytes,
                lay.total);
  HestonArgs a = {};
  a.steps = g->steps;
  char* base = (char*)ws;
  a.ckpt = base + lay.ckpt;
  a.part = (double*)(base + lay.part);
  a.paths = g->paths;
  a.nsteps = g->nsteps;
  a.payoff = g->payoff;
  a.lx0 = log(g->x0);
  a.x0 = g->x0;
  a.r = g->r;
  a.sig = g->sigma;
  a.k = g->k;
  a.th = g->theta;
  a.xi = g->xi;
  a.rho = g->rho;
  a.rhoc = sqrt(1.0 - g->rho * g->rho);
  a.y0 = g->y0;
  a.strike = g->strike;
  a.maturity = g->maturity;
  a.disc = exp(-g->r * g->maturity);
  a.k0 = g->key[0];
  a.k1 = g->key[1];
  a.epoch = g->epoch;
  hipStream_t st = (hipStream_t)stream;
  const unsigned nb = blocks_for(g->paths);
  double* sum_ds = (double*)(base + lay.sum);
  if (g->dtype == SDEGPU_F32) {
    float* tab = (float*)(base + lay.tab);
    hipLaunchKernelGGL(k_heston_table<float>, dim3(1), dim3(kBlock), 0, st, (const float*)g->steps,
                       g->nsteps, g->r, g->sigma, g->k, g->theta, g->xi, kGaussFold<float>, tab,
                       sum_ds);
    if (int e = launch_status("k_heston_table")) return e;
    if (v64) {
      // the variance's constants from the same FP32 (ds, sqrt ds), in FP64
      double* tabv = (double*)(base + lay.tabv);
      hipLaunchKernelGGL((k_heston_table<float, double>), dim3(1), dim3(kBlock), 0, st,
                         (const float*)g->steps, g->nsteps, g->r, g->sigma, g->k, g->theta, g->xi,
                         kGaussFold<float>, tabv, sum_ds);
      if (int e = launch_status("k_heston_table")) return e;
      if (g->method == 1)
        hipLaunchKernelGGL((k_heston_tangent<float, double>), dim3(nb), dim3(kBlock), 0, st, a,
                           (const float*)tab, (const double*)tabv, (const double*)sum_ds);
      else
        hipLaunchKernelGGL((k_heston_adjoint_seg<float, double, kHestonSeg64>), dim3(nb), dim3(kBlock),
                           0, st, a, (const float*)tab, (const double*)tabv,
                           (const double*)sum_ds);
    } else if (g->method == 1) {
      hipLaunchKernelGGL((k_heston_tangent<float, float>), dim3(nb), dim3(kBlock), 0, st, a,
                         (const float*)tab, (const float*)tab, (const double*)sum_ds);
    } else {
      // KEY1ST pays where the grid refills every SIMD (256 CUs of 8 blocks): 1M paths
      // as fast either way, 4M x 365 3.16 ms so and 3.19 without, 30,000 x 660 341 us so
      // and 325 without
      auto kernel = nb > 8192 ? k_heston_adjoint<kHestonSeg, true> : k_heston_adjoint<kHestonSeg, false>;
      hipLaunchKernelGGL(kernel, dim3(nb), dim3(kBlock), 0, st, a, (const float*)tab,
                         (float*)a.ckpt, (const double*)sum_ds);
    }
  } else {
    double* tab = (double*)(base + lay.tab);
    hipLaunchKernelGGL(k_heston_table<double>, dim3(1), dim3(kBlock), 0, st,
                       (const double*)g->steps, g->nsteps, g->r, g->sigma, g->k, g->theta, g->xi,
                       kGaussFold<double>, tab, sum_ds);
    if (int e = launch_status("k_heston_table")) return e;
    if (g->method == 1)
      hipLaunchKernelGGL((k_heston_tangent<double, double>), dim3(nb), dim3(kBlock), 0, st, a,
                         (const double*)tab, (const double*)tab, (const double*)sum_ds);
    else
      hipLaunchKernelGGL((k_heston_adjoint_seg<double, double, kHestonSeg64>), dim3(nb), dim3(kBlock),
                         0, st, a, (const double*)tab, (const double*)tab,
                         (const double*)sum_ds);
  }
  if (int e = launch_status(g->method == 1 ? "k_heston_tangent" : "k_heston_adjoint")) return e;
  return sum_columns(a.part, (int64_t)nb, kHestonNS, out, st);
}

extern "C" size_t sdegpu_loglin_greeks_workspace(int64_t paths) {
  if (paths < 1) return 0;
  return (size_t)blocks_for(paths) * kLogNS * sizeof(double);
}

extern "C" int sdegpu_loglin_greeks_run(const sdegpu_loglin_greeks* g, double* out, void* ws,
                                        size_t ws_bytes, void* stream) {
  if (!g || !out) return fail(SDEGPU_EINVAL, "loglin_greeks: null argument");
  if (g->dtype != SDEGPU_F32 && g->dtype != SDEGPU_F64)
    return fail(SDEGPU_EUNSUPPORTED, "loglin_greeks: dtype code %d", g->dtype);
  if (g->paths < 1 || g->paths > kMaxPaths || g->nsteps < 1 || !g->steps)
    return fail(SDEGPU_EINVAL, "loglin_greeks: paths=%lld steps=%d", (long long)g->paths,
                g->nsteps);
  if (!(g->x0 > 0.0)) return fail(SDEGPU_EINVAL, "loglin_greeks: need x0 > 0");
  if (g->payoff != 0 && g->payoff != 1)
    return fail(SDEGPU_EINVAL, "loglin_greeks: payoff kind %d", g->payoff);
  const size_t need = sdegpu_loglin_greeks_workspace(g->paths);
  if (!ws || ws_bytes < need)
    return fail(SDEGPU_ENOMEM, "loglin_greeks: workspace of %zu bytes, %zu needed", ws_bytes, need);
  LogArgs a = {};
  a.steps = g->steps;
  a.pois = g->pois;
  a.part = (double*)ws;
  a.paths = g->paths;
  a.nsteps = g->nsteps;
  a.payoff = g->payoff;
  a.lx0 = log(g->x0);
  a.x0 = g->x0;
  a.mu = g->mu;
  a.sig = g->sigma;
  a.ja = g->a;
  a.jb = g->b;
  a.strike = g->strike;
  a.maturity = g->maturity;
  a.disc = exp(-g->r * g->maturity);
  a.kw0 = g->key_w[0];
  a.kw1 = g->key_w[1];
  a.ew = g->epoch_w;
  a.kj0 = g->key_j[0];
  a.kj1 = g->key_j[1];
  a.ej = g->epoch_j;
  hipStream_t st = (hipStream_t)stream;
  const unsigned nb = blocks_for(g->paths);
  if (g->dtype == SDEGPU_F32)
    hipLaunchKernelGGL(k_loglin_greeks<float>, dim3(nb), dim3(kBlock), 0, st, a,
                       (const float*)a.steps, a.pois);
  else
    hipLaunchKernelGGL(k_loglin_greeks<double>, dim3(nb), dim3(kBlock), 0, st, a,
                       (const double*)a.steps, a.pois);
  if (int e = launch_status("k_loglin_greeks")) return e;
  return sum_columns(a.part, (int64_t)nb, kLogNS, out, st);
}
