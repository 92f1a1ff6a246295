// Euler path kernel for one coupled block of more than 8 working components
// (k_euler_wide): a dw correlated over 9..64 components, a Heston state of 5..32
// (log x, y) pairs on its last axis, a Hull-White value of 9..64 factors.
// sdepy draws such a block with one multivariate normal of any size
// (wiener_source.__call__, infrastructure.py:1524-1553) and steps it with the
// same euler_next update as any other state (integration.py:707-723).
//
// W waves share 64 paths.  Per step they draw the block's normals together, one
// Philox block of 4 after the other, into LDS, and after a barrier each applies
// the correlation and steps the components that it holds, at most R per lane.
// The step's table row is fetched a step ahead and spread out in LDS as a square
// with zeros above the diagonal.
//
// FP64: a wave holds 16 paths, a lane one component in four of one path, and
// v_mfma_f64_4x4x4 multiplies four rows of the square by four normals of the 16
// paths.  Its operands are one 8-byte LDS read each, 512 bytes for 256
// multiply-adds; as 16-byte broadcasts to lanes of 64 paths the coefficients
// took 1024 bytes for 128, and the kernel was bound by those reads.  Now the vector
// units are at work 62% of the time, the LDS 54%, the matrix cores 13%, and the
// waves wait 42% of theirs, for the LDS and at the two barriers of a step (20
// correlated lognormals, 100,000 paths x 252).
// FP32: a wave holds components (Heston: pairs) w, w + W, w + 2 W, ... of all 64
// paths and reads its coefficients as 16-byte broadcasts, four at a time, at
// fixed offsets (with scalar loads and a wait per piece of a row it took
// twice as long).
// One lane per path with the whole state, which both replace, took up to
// 256 registers, one or two waves per SIMD.  100 steps: 20 correlated lognormals
// FP64, 100,000 paths, 1010 us so, 680 with broadcasts, 553 now; 64 of
// them, 20,000 paths, 4880, 1140 and 656; FP32 12 of them, 200,000 paths, 680 and 280.
//
// The block's width m is a run-time value.  The kernel does everything the
// general k_euler instance does (component groups, recorded increments,
// antithetic halves, per-path parameters, correlation tables that change in
// time, the jump laws and the jump information, the backward pass) except the
// fused row moments and the deferred jump form: the jumps are summed in place,
// in sdepy's order.
//
// Correlation: dw = L z sqrt|ds| with the packed Cholesky rows of the step,
// row i summed over j = 0..i in order (FP64: four at a time), as in k_euler; the sum runs on over the zeros
// of the square (of the coefficients and of the normals past the width).
#pragma once
#include "euler_kernel.hpp"

namespace sdegpu {

template <bool B>
struct Flag {
  static constexpr bool value = B;
};

// FP64 applies the correlation on the matrix cores, with v_mfma_f64_4x4x4: four
// components by 16 paths, of four normals each.
template <typename T>
constexpr bool kWideMat = sizeof(T) == 8;

// The square of one row's coefficients: N rows and columns, the columns
// padded to whole 16-byte reads (FP64: against bank conflicts of its 4 x 4
// pieces, whose rows must not lie a multiple of 128 bytes apart).
template <typename T, int N>
struct WideSquare {
  static constexpr int CK = 16 / sizeof(T);  // coefficients per LDS read
  static constexpr int COLS = kWideMat<T> ? N + (N % 16 == 0 ? 4 : 0) : (N + CK - 1) / CK * CK;
  static constexpr int SIZE = N * COLS;
};

// Waves per SIMD that the compiler has to leave registers for.  A wave waits at
// two barriers a step, and what hides that are the other blocks of the CU: as
// many as the LDS has room for, or fewer where the registers would be
// spilled.  20 correlated lognormals FP64, 100,000 x 100: 4, 5, 6, 7 waves 593, 593, 599, 560
// us; 40 of them, 40,000 x 100: 685, 683, 603, (no room) 687; FP32 4
// and 6 waves: 502 and 412.  Jumps FP64, 40 of 40,000 x 100: 4, 5 waves 1601, 2159.
template <int MODEL, typename T, int W, int R, bool GEN>
constexpr int wide_occupancy() {
  constexpr bool jump = MODEL == SDEGPU_MODEL_JUMPDIFF, heston = MODEL == SDEGPU_MODEL_HESTON;
  if (!kWideMat<T>) return W == 6 ? (jump ? 5 : 6) : W == 3 && (heston || (jump && R == 7)) ? 5 : 4;
  if (jump) return W == 4 && !GEN ? 5 : R == 8 ? 2 : 4;
  if (GEN || (heston ? W * R == 32 : W * R == 64)) return 4;
  return W == 4 && R < 6 && !heston ? 7 : 6;
}

// GEN: recorded increments, per-path parameters and per-path intensities.
//
// STREAM: rows begin on 64-byte lines, and the stores stream past the L2.
// Where they don't, every wave's 64 values share their first and last line with the
// neighbouring blocks', and streamed one by one those halves are
// written back alone: 400,003 paths of 12 FP32 OU components x 13, 14 rows 161 us, 81 by
// plain stores that the L2 joins (400,000 paths: 81 and 83; 1,636,947: 631 and 307).  So that
// neighbours meet in one L2, XCD x (blockIdx.x mod 8) steps the x-th eighth of the blocks;
// without that the 1,636,947 paths take 492.  Streamed rows are 1 to 2% slower in that order.
template <int MODEL, typename T, int W, int R, bool GEN, bool STREAM>
__global__ __launch_bounds__(64 * W, (wide_occupancy<MODEL, T, W, R, GEN>())) void k_euler_wide(const EulerArgs a,
                                                       const T* __restrict__ coef,
                                                       const int32_t* __restrict__ store_row,
                                                       const double* __restrict__ pois,
                                                       T* __restrict__ out) {
  constexpr bool kJump = MODEL == SDEGPU_MODEL_JUMPDIFF;
  constexpr bool kHeston = MODEL == SDEGPU_MODEL_HESTON;
  constexpr bool kOU = MODEL == SDEGPU_MODEL_OU;
  constexpr bool kMat = kWideMat<T>;
  constexpr int N = R * W;
  using Sq = WideSquare<T, N>;
  constexpr int CK = Sq::CK, COLS = Sq::COLS;
  constexpr int NS = kHeston ? 3 : 1;  // squares: of log x (or all); y by x, y by y
  constexpr int NB = kHeston ? 2 : 1;  // normals' buffers: of log x (or all), of y
  constexpr int NPAR = 5 * N;
  // the squares, then ds, sqrt|ds| and the parameter blocks
  constexpr int NTAB = NS * Sq::SIZE + 2 + NPAR;
  __shared__ __align__(16) T chol[NTAB];
  T* const par_lds = chol + NS * Sq::SIZE;
  __shared__ T z[NB][COLS][64];
  __shared__ uint32_t words[kJump ? N : 1][kJump ? 64 : 1];

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // the block's place among the paths (the last few, past whole eighths, keep theirs)
  const unsigned eighth = STREAM ? 0u : gridDim.x >> 3;
  const unsigned blk = blockIdx.x < 8u * eighth ? (blockIdx.x & 7u) * eighth + (blockIdx.x >> 3)
                                                : blockIdx.x;
  // A lane draws for path `lane` of the block and steps the state of path `pl`.
  const int quad = lane >> 4;
  const int pl = kMat ? 16 * (w & 3) + (lane & 15) : lane;
  // where a row of z holds a path's value (FP64: two of the four rows that the
  // matrix instruction reads at once would meet in the same banks)
  auto col = [&](int v, int p) { return kMat ? p ^ ((v & 1) << 4) : p; };
  const int m = a.nvars;
  const int n = kHeston ? m / 2 : m;  // width of a parameter block
  gauss_init<T>(64 * W);
  const bool replay = GEN && a.replay_dw != nullptr;
  const bool replay_j = GEN && a.replay_dj != nullptr;
  const bool pp = GEN && a.ppar != nullptr;
  const uint32_t zero_below = kJump && !(GEN && (a.replay_dj || a.lamp))
                                  ? zero_count_bound(pois, (int64_t)a.nsteps * m, 64 * W)
                                  : 0u;
  for (int i = threadIdx.x; i < NTAB; i += 64 * W) chol[i] = (T)0;
  for (int i = threadIdx.x; i < NB * COLS * 64; i += 64 * W) (&z[0][0][0])[i] = (T)0;

  // Table element e of a step: the header and the parameters go to par_lds, the
  // triangle's (i, j) to its square.  Thread t moves elements t, t + 64 W, ...
  constexpr int MAXC = 2 + (kHeston ? 2 * N * (2 * N + 1) / 2 : N * (N + 1) / 2) + NPAR;
  constexpr int NE = (MAXC + 64 * W - 1) / (64 * W);
  const int ncoef = a.ncoef < a.poff + 5 * n ? a.ncoef : a.poff + 5 * n;
  int dst[NE];  // its place in chol (-1: none)
#pragma unroll
  for (int k = 0; k < NE; ++k) {
    const int e = k * 64 * W + (int)threadIdx.x;
    dst[k] = -1;
    if (e >= ncoef) continue;
    if (e < 2) {
      dst[k] = NS * Sq::SIZE + e;
    } else if (e >= a.poff) {
      const int b = (e - a.poff) / n;
      dst[k] = NS * Sq::SIZE + 2 + b * N + (e - a.poff - b * n);
    } else {
      // row i holds elements i (i + 1) / 2 .. of the packed triangle
      const int q = e - 2;
      int i = (int)((sqrtf(8.f * (float)q + 1.f) - 1.f) * .5f);
      while ((i + 1) * (i + 2) / 2 <= q) ++i;
      while (i * (i + 1) / 2 > q) --i;
      const int j = q - i * (i + 1) / 2;
      if (!kHeston || i < n)
        dst[k] = i * COLS + j;
      else if (j < n)
        dst[k] = Sq::SIZE + (i - n) * COLS + j;
      else
        dst[k] = 2 * Sq::SIZE + (i - n) * COLS + (j - n);
    }
  }
  T ahead[NE];
  auto fetch = [&](int s) {
#pragma unroll
    for (int k = 0; k < NE; ++k)
      if (dst[k] >= 0) ahead[k] = coef[(int64_t)s * a.ncoef + k * 64 * W + (int)threadIdx.x];
  };

  const int64_t P = a.paths;
  const int64_t tid = (int64_t)blk * 64 + pl;
  // lanes beyond the last path step a copy of it and store nothing
  const bool live = tid < P;
  const int64_t gid = live ? tid : P - 1;
  auto jump_path = [&](int64_t i) {
    return (uint32_t)(a.anti_j > 0 && i >= a.anti_j ? i - a.anti_j : i);
  };
  const uint32_t path_j = jump_path(gid);
  // the path that the lane draws for
  const int64_t did = min((int64_t)blk * 64 + lane, P - 1);
  const bool flip_w = a.anti_w > 0 && did >= a.anti_w;
  const uint32_t path_w = (uint32_t)(flip_w ? did - a.anti_w : did);
  const uint32_t path_p = jump_path(did);
  const int64_t mt = a.m_total, c0 = a.comp0;
  const int64_t mtb = kHeston ? mt / 2 : mt, c0b = kHeston ? c0 / 2 : c0;
  const T* __restrict__ ppar = (const T*)a.ppar;
  const T* __restrict__ x0p = (const T*)a.x0_paths;
  auto x0_of = [&](int v) -> T {
    return x0p ? x0p[(c0 + v) * P + gid] : (T)a.x0[v];
  };
  // the r-th component of the wave (FP64: of the lane), and whether there is one; rows
  // without one step zeros
  auto comp = [&](int r) { return kMat ? r * W + (w >> 2) * 4 + quad : r * W + w; };
  auto has = [&](int r) { return comp(r) < n; };
  // parameter block b of component (Heston: pair) v at a step (per path: at the
  // step's offset pbase into ppar)
  int64_t pbase = 0;
  auto par = [&](int b, int v) -> T {
    if (pp) return v < n ? ppar[pbase + ((int64_t)b * mtb + c0b + v) * P + gid] : (T)0;
    return par_lds[2 + b * N + v];
  };

  T x[R];  // log x for Heston
  T vy[kHeston ? R : 1];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    x[r] = has(r) ? x0_of(comp(r)) : (T)0;
    if constexpr (kHeston) vy[r] = has(r) ? x0_of(n + comp(r)) : (T)0;
  }
  int cnt[R];
#pragma unroll
  for (int r = 0; r < R; ++r) cnt[r] = 0;
  int interval_jumps = 0;

  auto put = [&](T v, T* at) {
    if constexpr (STREAM)
      __builtin_nontemporal_store(v, at);
    else
      *at = v;
  };
  // Every thread of the block must call it.
  auto store = [&](int row) {
    T* o_row = out + ((int64_t)row * a.out_stride + a.out0) * P + gid;
    if (kOU && a.out_group != 1) {
      // hull_white_SDE.let: the sum over the block's factors (out_group = m),
      // in order, from the waves' values in the normals' buffer
      __syncthreads();
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (has(r)) z[0][comp(r)][pl] = x[r];
      __syncthreads();
      if (w == 0 && (int64_t)blk * 64 + lane < P) {
        T val = (T)0;
        for (int v = 0; v < m; ++v) val = val + z[0][v][lane];
        put(val, o_row - gid + did);
      }
      return;
    }
    if (!live) return;
    T* o = o_row + comp(0) * P;  // row r of the wave is r W components further on
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (!has(r)) break;
      if constexpr (kHeston) {
        put((T)exp(x[r]), o);
        if (a.nout == m) put(vy[r], o + n * P);
      } else if (comp(r) < a.nout) {
        T val = x[r];
        if constexpr (OutRule<MODEL>::exp_all) val = exp(val);
        put(val, o);
      }
      o += W * P;
    }
  };

  // The flat indices g .. g+m-1 of a stream lie in Philox blocks g/4 ...; f
  // gets a block and the component of its first value, every wave each W-th one.
  // FP32: the waves take turns at the first, as those that draw one more would
  // otherwise run on the same SIMD (3 to 10% faster; FP64 is 1 to 3% slower so).
    int turn = kMat ? w : (int)((blockIdx.x + (unsigned)w) % (unsigned)W);
  auto each_block = [&](uint64_t g, int first, auto f) {
    const uint32_t b0 = (uint32_t)(g >> 2);
    const int off = (int)(g & 3u);
    const int nb = (off + m + 3) >> 2;
    for (int i = 0; i * W < nb; ++i) {
      const int q = i * W + first;
      if (q >= nb) break;
      f(b0 + q, 4 * q - off);
    }
  };

  // acc[r] += sum over columns of square[row of r][column] zz[column]; of a
  // triangle only the columns up to the rows r of any wave.
  auto apply = [&](T(&acc)[R], const T* square, const T(*zz)[64], auto triangle) {
    if constexpr (kMat) {
      // lane 16 k + 4 b + i holds element (i, k) of the four rows' piece, for
      // each b, and the normal k of path 16 k + 4 b + j; the sum of component i
      // of a path comes out in lane 16 i + 4 b + j
      constexpr int H = W / 4;
      const T* mine = square + ((w >> 2) * 4 + (lane & 3)) * COLS + quad;
#pragma unroll
      for (int c = 0; c < N / 4; ++c) {
        const T zc = zz[4 * c + quad][col(quad, pl)];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          if (decltype(triangle)::value && (r + 1) * H <= c) continue;
          acc[r] = __builtin_amdgcn_mfma_f64_4x4x4f64(mine[r * W * COLS + 4 * c], zc, acc[r], 0,
                                                      0, 0);
        }
      }
      return;
    }
    const T* mine = square + w * COLS;
#pragma unroll
    for (int q = 0; q < COLS / CK; ++q) {
      T zc[CK];
#pragma unroll
      for (int l = 0; l < CK; ++l) zc[l] = zz[q * CK + l][lane];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (decltype(triangle)::value && (r + 1) * W <= q * CK) continue;
        T cf[CK];
        __builtin_memcpy(cf, __builtin_assume_aligned(mine + r * W * COLS + q * CK, 16), 16);
#pragma unroll
        for (int l = 0; l < CK; ++l) acc[r] = acc[r] + cf[l] * zc[l];
      }
    }
  };

  if (a.nsteps > 0) fetch(0);
  __syncthreads();
  if (a.row0 >= 0) store(a.row0);
  __syncthreads();

  for (int s = 0; s < a.nsteps; ++s) {
    const uint64_t g = (uint64_t)s * mt + c0;  // flat index of the block's first normal
    pbase = (int64_t)s * a.ppar_step;
    const T* rp = replay ? (const T*)a.replay_dw + (int64_t)g * P + gid : nullptr;

    // the step's table row, normals and Poisson words into LDS
#pragma unroll
    for (int k = 0; k < NE; ++k)
      if (dst[k] >= 0) chol[dst[k]] = ahead[k];
    if (!replay) {
      each_block(g, turn, [&](uint32_t blk, int v0) {
        T zz[4];
        normals4<T>(blk, path_w, a.c2w, a.ew, a.kw0, a.kw1, zz);
#pragma unroll
        for (int l = 0; l < 4; ++l) {
          const int v = v0 + l;
          const T val = flip_w ? -zz[l] : zz[l];
          if (v >= 0 && v < m) {
            if (!kHeston || v < n)
              z[0][v][col(v, lane)] = val;
            else
              z[NB - 1][v - n][col(v - n, lane)] = val;
          }
        }
      });
    }
    if constexpr (kJump) {
      if (!replay_j) {
        each_block(g, kMat ? w : W - 1 - turn, [&](uint32_t blk, int v0) {
          const ctr4 u = philox4x32_10(ctr4{blk, path_p, a.c2p, a.ej}, a.kj0, a.kj1);
          const uint32_t uu[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
          for (int l = 0; l < 4; ++l)
            if (v0 + l >= 0 && v0 + l < m) words[v0 + l][lane] = uu[l];
        });
      }
    }
    if constexpr (!kMat) turn = turn + 1 < W ? turn + 1 : 0;
    __syncthreads();
    if (s + 1 < a.nsteps) fetch(s + 1);
    const int row = store_row[s];
    const T ds = par_lds[0], sq = par_lds[1];

    if constexpr (kHeston) {
      // dw of the log-x values (zx) and of the variances (zy)
      T zx[R], zy[R];
#pragma unroll
      for (int r = 0; r < R; ++r) zx[r] = zy[r] = (T)0;
      if (replay) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
          if (has(r)) {
            zx[r] = rp[(int64_t)comp(r) * P];
            zy[r] = rp[(int64_t)(n + comp(r)) * P];
          }
        }
      } else {
        if (a.has_corr) {
          // the y rows: every column of log x, then the triangle of y
          apply(zx, chol, z[0], Flag<true>{});
          apply(zy, chol + Sq::SIZE, z[0], Flag<false>{});
          apply(zy, chol + 2 * Sq::SIZE, z[NB - 1], Flag<true>{});
        } else {
#pragma unroll
          for (int r = 0; r < R; ++r) {
            zx[r] = z[0][comp(r)][col(comp(r), pl)];
            zy[r] = z[NB - 1][comp(r)][col(comp(r), pl)];
          }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
          zx[r] = zx[r] * sq;
          zy[r] = zy[r] * sq;
        }
      }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int v = comp(r);
        heston_next<T>(x[r], vy[r], cnt[r], par(0, v), par(1, v), par(2, v), par(3, v),
                       par(4, v), ds, zx[r], zy[r]);
      }
    } else {
      // OU with correlations and table parameters: sigma_i sqrt|ds| is folded
      // into the Cholesky rows by the host, as for k_euler
      const bool ou_folded = kOU && a.has_corr && !replay && !pp;
      T dw[R];
#pragma unroll
      for (int r = 0; r < R; ++r)
        dw[r] = ou_folded ? fma(par(0, comp(r)), x[r], par(1, comp(r))) : (T)0;
      if (replay) {
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (has(r)) dw[r] = rp[(int64_t)comp(r) * P];
      } else if (a.has_corr) {
        apply(dw, chol, z[0], Flag<true>{});
        if (!ou_folded) {
#pragma unroll
          for (int r = 0; r < R; ++r) dw[r] = dw[r] * sq;
        }
      } else {
#pragma unroll
        for (int r = 0; r < R; ++r) dw[r] = z[0][comp(r)][col(comp(r), pl)] * sq;
      }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int v = comp(r);
        if constexpr (MODEL == SDEGPU_MODEL_WIENER || MODEL == SDEGPU_MODEL_LOGNORM) {
          x[r] = x[r] + (par(0, v) * ds + par(1, v) * dw[r]);
        } else if constexpr (kOU) {
          if (ou_folded) {
            x[r] = dw[r];
          } else {
            const T av = pp ? fma(-par(0, v), ds, (T)1) : par(0, v);
            const T bv = pp ? par(1, v) * ds : par(1, v);
            x[r] = av * x[r] + (bv + par(2, v) * dw[r]);
          }
        } else if constexpr (MODEL == SDEGPU_MODEL_CIR) {
          x[r] = cir_next<T>(x[r], par(0, v), par(1, v), par(2, v), ds, dw[r]);
        } else if constexpr (kJump) {
          T inc = par(0, v) * ds + par(1, v) * dw[r];
          if (replay_j) {
            if (has(r)) inc = inc + ((const T*)a.replay_dj)[((int64_t)g + v) * P + gid];
          } else if (has(r)) {
            const uint32_t word = words[v][pl];
            if (word >= zero_below) {
              const double* pq = pois + ((int64_t)s * m + v) * 2;
              double lamds = pq[0], p0 = pq[1];
              if (GEN && a.lamp) {
                // per-path intensity: pois holds |ds|
                lamds = a.lamp[(int64_t)s * a.lamp_step + (c0 + v) * P + gid] * lamds;
                p0 = exp(-lamds);
              }
              const int nj = poisson_inv(u01_f64(word), lamds, p0, kPoissonCap);
              if (nj > 0) {
                const bool neg = ds < (T)0;
                const T* pj = par_lds + 2;
                const T p2 = a.jump_law == SDEGPU_JUMP_NORMAL ? (T)0 : pj[4 * N + v];
                const T acc = jump_total<T>(a.jump_law, nj, (uint32_t)(g + v), path_j, a.c2j,
                                            a.ej, a.kj0, a.kj1, pj[2 * N + v], pj[3 * N + v],
                                            p2);
                inc = inc + (neg ? -acc : acc);
                cnt[r] += neg ? -nj : nj;
                interval_jumps += neg ? -nj : nj;
              }
            }
          }
          x[r] = x[r] + inc;
        }
      }
    }

    if (row >= 0) {
      store(row);
      if constexpr (kJump) {
        if (a.info_rows) add_interval_jumps(a, row, live, interval_jumps);
        interval_jumps = 0;
      }
    }
    __syncthreads();
  }

  if (a.info_paths && (kHeston || kJump) && live) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (has(r)) a.info_paths[(c0b + comp(r)) * P + gid] = cnt[r];
  }
}

// wiener_source.__call__ for one correlated block of m <= W components (see
// k_wiener_fill): dz = L z sqrt|ds| with the rows summed in order.
template <typename T, int W>
__global__ __launch_bounds__(kBlock) void k_wiener_fill_wide(
    uint32_t k0, uint32_t k1, uint32_t epoch, uint32_t c2, int64_t paths, int64_t nslots,
    const T* __restrict__ coef, int ncoef, int has_corr, int m, int comp0, int m_total,
    T* __restrict__ out) {
  gauss_init<T>();
  const int64_t gid = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (gid >= paths) return;
  const uint32_t path = (uint32_t)gid;
  for (int64_t s = 0; s < nslots; ++s) {
    T z[W];
    normals_span<T, W>((uint64_t)s * m_total + comp0, m, path, c2, epoch, k0, k1, z);
    const T* c = coef + s * ncoef;
    const T sq = c[1];
    T* o = out + (s * m_total + comp0) * paths + gid;
    if (has_corr) {
      const T* L = c + 2;
#pragma unroll
      for (int i = W - 1; i >= 0; --i) {
        if (i < m) {
          const T* Li = L + i * (i + 1) / 2;
          T acc = (T)0;
#pragma unroll
          for (int j = 0; j <= i; ++j) acc = acc + Li[j] * z[j];
          o[i * paths] = acc * sq;
        }
      }
    } else {
#pragma unroll
      for (int v = 0; v < W; ++v)
        if (v < m) o[v * paths] = z[v] * sq;
    }
  }
}

// Waves that share 64 paths and components (Heston: pairs) per wave for a width:
// the smallest of the instantiated shapes that holds it.
struct WideShape {
  int waves, rows;
};
template <typename T>
inline WideShape wide_shape(int model, int m) {
  const bool h = model == SDEGPU_MODEL_HESTON;
  const int n = h ? m / 2 : m;
  if (kWideMat<T>) {
    // 4 waves hold 4 components of 16 paths each per row, 8 waves twice that
    const int rows = (n + 3) / 4, most = h ? 4 : 6;
    if (rows > 16 || (h && rows > 8)) return WideShape{0, 0};
    if (rows <= most) return WideShape{4, rows < (h ? 2 : 3) ? (h ? 2 : 3) : rows};
    return WideShape{8, h ? (rows + 1) / 2 : rows <= 8 ? 4 : rows <= 12 ? 6 : 8};
  }
  const WideShape all[2][7] = {{{2, 6}, {2, 8}, {3, 7}, {3, 8}, {4, 8}, {6, 8}, {8, 8}},
                               {{2, 3}, {2, 4}, {3, 4}, {4, 4}, {6, 4}, {8, 4}, {8, 4}}};
  for (const WideShape& s : all[h ? 1 : 0])
    if (s.waves * s.rows >= n) return s;
  return WideShape{0, 0};
}

// k_euler_wide and k_wiener_fill_wide instances (euler_wide_f32.hip,
// euler_wide_f64.hip): the kernel for a model and a width of 9..64, or null.
// Blocks of 64 * wide_shape<T>(model, m).waves threads, one per 64 paths; gen: recorded
// increments, per-path parameters or intensities (plain stores only); stream: rows of whole 64-byte lines.
template <typename T>
EulerKernel<T> euler_wide_kernel(int model, int m, bool gen, bool stream);

template <typename T>
using WienerFillWide = void (*)(uint32_t, uint32_t, uint32_t, uint32_t, int64_t, int64_t,
                                const T*, int, int, int, int, int, T*);
template <typename T>
WienerFillWide<T> wiener_fill_wide_kernel(int m);
template <>
EulerKernel<float> euler_wide_kernel<float>(int model, int m, bool gen, bool stream);
template <>
EulerKernel<double> euler_wide_kernel<double>(int model, int m, bool gen, bool stream);
template <>
WienerFillWide<float> wiener_fill_wide_kernel<float>(int m);
template <>
WienerFillWide<double> wiener_fill_wide_kernel<double>(int m);

template <int MODEL, typename T, bool GEN, bool STREAM>
EulerKernel<T> pick_wide(int m) {
  const WideShape s = wide_shape<T>(MODEL, m);
  const int key = s.waves * 16 + s.rows;
  if constexpr (MODEL == SDEGPU_MODEL_HESTON && kWideMat<T>) {
    switch (key) {
      case 4 * 16 + 2: return k_euler_wide<MODEL, T, 4, 2, GEN, STREAM>;
      case 4 * 16 + 3: return k_euler_wide<MODEL, T, 4, 3, GEN, STREAM>;
      case 4 * 16 + 4: return k_euler_wide<MODEL, T, 4, 4, GEN, STREAM>;
      case 8 * 16 + 3: return k_euler_wide<MODEL, T, 8, 3, GEN, STREAM>;
      case 8 * 16 + 4: return k_euler_wide<MODEL, T, 8, 4, GEN, STREAM>;
      default: return nullptr;
    }
  } else if constexpr (MODEL == SDEGPU_MODEL_HESTON) {
    switch (key) {
      case 2 * 16 + 3: return k_euler_wide<MODEL, T, 2, 3, GEN, STREAM>;
      case 2 * 16 + 4: return k_euler_wide<MODEL, T, 2, 4, GEN, STREAM>;
      case 3 * 16 + 4: return k_euler_wide<MODEL, T, 3, 4, GEN, STREAM>;
      case 4 * 16 + 4: return k_euler_wide<MODEL, T, 4, 4, GEN, STREAM>;
      case 6 * 16 + 4: return k_euler_wide<MODEL, T, 6, 4, GEN, STREAM>;
      case 8 * 16 + 4: return k_euler_wide<MODEL, T, 8, 4, GEN, STREAM>;
      default: return nullptr;
    }
  } else if constexpr (kWideMat<T>) {
    switch (key) {
      case 4 * 16 + 3: return k_euler_wide<MODEL, T, 4, 3, GEN, STREAM>;
      case 4 * 16 + 4: return k_euler_wide<MODEL, T, 4, 4, GEN, STREAM>;
      case 4 * 16 + 5: return k_euler_wide<MODEL, T, 4, 5, GEN, STREAM>;
      case 4 * 16 + 6: return k_euler_wide<MODEL, T, 4, 6, GEN, STREAM>;
      case 8 * 16 + 4: return k_euler_wide<MODEL, T, 8, 4, GEN, STREAM>;
      case 8 * 16 + 6: return k_euler_wide<MODEL, T, 8, 6, GEN, STREAM>;
      case 8 * 16 + 8: return k_euler_wide<MODEL, T, 8, 8, GEN, STREAM>;
      default: return nullptr;
    }
  } else {
    switch (key) {
      case 2 * 16 + 6: return k_euler_wide<MODEL, T, 2, 6, GEN, STREAM>;
      case 2 * 16 + 8: return k_euler_wide<MODEL, T, 2, 8, GEN, STREAM>;
      case 3 * 16 + 7: return k_euler_wide<MODEL, T, 3, 7, GEN, STREAM>;
      case 3 * 16 + 8: return k_euler_wide<MODEL, T, 3, 8, GEN, STREAM>;
      case 4 * 16 + 8: return k_euler_wide<MODEL, T, 4, 8, GEN, STREAM>;
      case 6 * 16 + 8: return k_euler_wide<MODEL, T, 6, 8, GEN, STREAM>;
      case 8 * 16 + 8: return k_euler_wide<MODEL, T, 8, 8, GEN, STREAM>;
      default: return nullptr;
    }
  }
}

template <int MODEL, typename T>
EulerKernel<T> pick_wide(int m, bool gen, bool stream) {
  if (gen) return pick_wide<MODEL, T, true, false>(m);
  return stream ? pick_wide<MODEL, T, false, true>(m) : pick_wide<MODEL, T, false, false>(m);
}

#define SDEGPU_EULER_WIDE_SET(T)                                                         \
  template <>                                                                            \
  EulerKernel<T> euler_wide_kernel<T>(int model, int m, bool gen, bool stream) {         \
    if (m <= SDEGPU_MAX_VARS || m > SDEGPU_MAX_COUPLED) return nullptr;                  \
    switch (model) {                                                                     \
      case SDEGPU_MODEL_WIENER: return pick_wide<SDEGPU_MODEL_WIENER, T>(m, gen, stream);\
      case SDEGPU_MODEL_LOGNORM: return pick_wide<SDEGPU_MODEL_LOGNORM, T>(m, gen, stream);\
      case SDEGPU_MODEL_OU: return pick_wide<SDEGPU_MODEL_OU, T>(m, gen, stream);        \
      case SDEGPU_MODEL_CIR: return pick_wide<SDEGPU_MODEL_CIR, T>(m, gen, stream);      \
      case SDEGPU_MODEL_HESTON: return pick_wide<SDEGPU_MODEL_HESTON, T>(m, gen, stream);\
      case SDEGPU_MODEL_JUMPDIFF: return pick_wide<SDEGPU_MODEL_JUMPDIFF, T>(m, gen, stream);\
      default: return nullptr;                                                           \
    }                                                                                    \
  }                                                                                      \
  template <>                                                                            \
  WienerFillWide<T> wiener_fill_wide_kernel<T>(int m) {                                  \
    if (m <= SDEGPU_MAX_VARS || m > SDEGPU_MAX_COUPLED) return nullptr;                  \
    return m <= 16 ? k_wiener_fill_wide<T, 16>                                           \
                   : m <= 32 ? k_wiener_fill_wide<T, 32> : k_wiener_fill_wide<T, 64>;    \
  }

}  // namespace sdegpu
