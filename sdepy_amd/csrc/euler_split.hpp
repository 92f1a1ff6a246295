// Euler path kernel for runs of few paths (k_euler_split): several waves
// share 64 paths.
//
// k_euler gives each path one lane for the whole step loop, so a run of a few
// thousand paths leaves most of the chip's 1024 SIMDs without a wave, and its
// time is the serial chain of one: draw, step, store, step after step.  Of a
// step's instructions most do not depend on the state: the Philox draws,
// Box-Muller, the correlation, the drift of the additive models, the jumps and
// their sizes.  Here the W waves of a block draw the noise of different steps
// of the same 64 paths, a chunk of steps ahead, into LDS, and every
// wave then runs the short remaining recursion over all steps of the chunk
// (each holds the same state) and stores its share of the output rows, every
// W-th one.  So the exp and the stores of the rows are shared out too.  One
// barrier per chunk: the noise of the next chunk is drawn into the other
// buffer.
//
// The draws, counters and counts are k_euler's, and so is the arithmetic but
// for the order of the OU noise sum (x = a x + (b + noise)).  Takes the
// plain and the antithetic runs of up to 4 components (2 with jumps);
// recorded increments, component groups, per-path parameters or intensities and fused
// row moments stay with k_euler.
#pragma once
#include "euler_kernel.hpp"

namespace sdegpu {

// Units of CH steps (whole Philox blocks) per chunk, MOST of them (4 for the
// 3-component states, whose unit is 4 steps of 3 blocks): 8, so that 8 waves have
// one each.  FP64 jumps take 52 KB of LDS so, three blocks per CU: grids of
// more than three, whose blocks have 4 waves at most, run with 4 units and 28 KB.  FP64, 250
// steps, 251 rows: Kou of 60,000 paths 159 -> 142 us, two Mertons 310 -> 278; of
// 40,000 paths (2.4 blocks per CU) 114 with 8 units, 121 with 4.
template <int M, int MOST>
struct SplitChunk {
  static constexpr int U = Chunking<M>::NZ > 4 ? 4 : MOST;
  static constexpr int L = U * Chunking<M>::CH;
};

template <int K>
struct Count {
  static constexpr int value = K;
};

// STREAM: rows begin on 64-byte lines, and the stores stream past the L2.
// Where they don't, the halves of the lines that neighbouring blocks share are joined
// in the L2 (as in k_euler_wide): 4 OU components FP32 64,999 x 250, every step stored,
// 121 us alone, 162 streamed, 100 so; lognormal 162 and 98.  FP64 Heston and CIR, whose
// lines are further apart in time, are up to 20% slower so and always stream.
template <int MODEL, typename T, int M, int D, bool STREAM, int MOST = 8>
__global__ __launch_bounds__(64 * MOST) void k_euler_split(
    const EulerArgs a, const T* __restrict__ coef, const int32_t* __restrict__ store_row,
    const double* __restrict__ pois, T* __restrict__ out) {
  constexpr int CH = Chunking<M>::CH, NZ = Chunking<M>::NZ;
  constexpr int U = SplitChunk<M, MOST>::U, L = SplitChunk<M, MOST>::L;
  constexpr bool kJump = MODEL == SDEGPU_MODEL_JUMPDIFF;
  constexpr bool kHeston = MODEL == SDEGPU_MODEL_HESTON;
  constexpr bool kOU = MODEL == SDEGPU_MODEL_OU;
  constexpr bool kCIR = MODEL == SDEGPU_MODEL_CIR;
  constexpr int N = kHeston ? M / 2 : M;
  // noise[b][step][component][lane], jumps[b][step][component][lane]
  __shared__ T noise[2][L][M][64];
  __shared__ int jumps[kJump ? 2 : 1][kJump ? L : 1][kJump ? M : 1][kJump ? 64 : 1];

  // read into scalar registers here, or the compiler takes the block size for
  // a per-lane value and with it everything that depends on a wave's units
  const int W = __builtin_amdgcn_readfirstlane((int)(blockDim.x >> 6));
  gauss_init<T>(64 * W);
  const uint32_t zero_below =
      kJump ? zero_count_bound(pois, (int64_t)a.nsteps * M, 64 * W) : 0u;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t P = a.paths;
  // the block's place among the paths: XCD x takes the x-th eighth of the blocks (the last few,
  // past whole eighths, keep theirs)
  const unsigned eighth = STREAM ? 0u : gridDim.x >> 3;
  const unsigned blk = blockIdx.x < 8u * eighth ? (blockIdx.x & 7u) * eighth + (blockIdx.x >> 3)
                                                : blockIdx.x;
  const int64_t tid = (int64_t)blk * 64 + lane;
  // lanes beyond the last path step a copy of it and store nothing
  const bool live = tid < P;
  const int64_t gid = live ? tid : P - 1;
  const uint32_t path = (uint32_t)gid;
  const bool flip_w = a.anti_w > 0 && gid >= a.anti_w;
  const uint32_t path_w = flip_w ? (uint32_t)(gid - a.anti_w) : path;
  const uint32_t path_j = (a.anti_j > 0 && gid >= a.anti_j) ? (uint32_t)(gid - a.anti_j) : path;
  const int n = a.nsteps;

  T x[M];
  if (a.x0_paths) {
#pragma unroll
    for (int v = 0; v < M; ++v) x[v] = ((const T*)a.x0_paths)[v * P + gid];
  } else {
#pragma unroll
    for (int v = 0; v < M; ++v) x[v] = (T)a.x0[v];
  }
  int cnt[M];
#pragma unroll
  for (int v = 0; v < M; ++v) cnt[v] = 0;
  int interval_jumps = 0;
  auto store = [&](int row) {
    if (live)
      store_state<MODEL, T, M, D, false, false, STREAM>(out, a, row, x, gid, true, (T*)nullptr);
  };
  if (a.row0 >= 0 && w == 0) store(a.row0);

  // The state-independent part of the chunk's steps: wave w's units.
  auto draw = [&](int c0, int b) {
    // (counted from 0: a loop that starts at w loses the proof that its table
    // addresses are wave-uniform, and with it the scalar loads)
    for (int i = 0; i * W < U; ++i) {
      const int u = i * W + w;
      const int s0 = c0 + u * CH;
      if (u >= U || s0 >= n) break;
      T z[NZ];
      const uint32_t b0 = (uint32_t)(((int64_t)s0 * M) >> 2);
#pragma unroll
      for (int j = 0; j < NZ / 4; ++j)
        normals4<T>(b0 + j, path_w, a.c2w, a.ew, a.kw0, a.kw1, z + 4 * j);
      if (flip_w) {
#pragma unroll
        for (int i = 0; i < NZ; ++i) z[i] = -z[i];
      }
      uint32_t words[kJump ? NZ : 1];
      if constexpr (kJump) {
#pragma unroll
        for (int j = 0; j < NZ / 4; ++j) {
          const ctr4 r = philox4x32_10(ctr4{b0 + j, path_j, a.c2p, a.ej}, a.kj0, a.kj1);
          words[4 * j + 0] = r.x;
          words[4 * j + 1] = r.y;
          words[4 * j + 2] = r.z;
          words[4 * j + 3] = r.w;
        }
      }
#pragma unroll
      for (int k = 0; k < CH; ++k) {
        const int s = s0 + k;
        if (s >= n) break;
        const T* c = coef + (int64_t)s * a.ncoef;
        const T ds = c[0], sq = c[1];
        const T* p = c + a.poff;
        const bool folded = kOU && a.has_corr;  // sigma sqrt|ds| in the Cholesky rows
        T dw[M];
        if (a.has_corr) {
          const T* Lc = c + 2;
          int idx = 0;
#pragma unroll
          for (int i = 0; i < M; ++i) {
            T acc = kOU ? p[M + i] : (T)0;
#pragma unroll
            for (int j = 0; j <= i; ++j) acc = acc + Lc[idx++] * z[k * M + j];
            dw[i] = folded ? acc : acc * sq;
          }
        } else {
#pragma unroll
          for (int v = 0; v < M; ++v) dw[v] = z[k * M + v] * sq;
        }
#pragma unroll
        for (int v = 0; v < M; ++v) {
          T q = dw[v];
          if constexpr (kOU) {
            if (!folded) q = p[M + v] + p[2 * M + v] * dw[v];
          } else if constexpr (!kHeston && !kCIR) {
            q = p[v] * ds + p[M + v] * dw[v];
          }
          if constexpr (kJump) {
            int nj = 0;
            const uint32_t word = words[k * M + v];
            if (word >= zero_below) {
              const double* pq = pois + ((int64_t)s * M + v) * 2;
              nj = poisson_inv(u01_f64(word), pq[0], pq[1], kPoissonCap);
              if (nj > 0) {
                const T p2 = a.jump_law == SDEGPU_JUMP_NORMAL ? (T)0 : p[4 * M + v];
                const T acc = jump_total<T>(a.jump_law, nj, (uint32_t)((int64_t)s * M + v),
                                            path_j, a.c2j, a.ej, a.kj0, a.kj1, p[2 * M + v],
                                            p[3 * M + v], p2);
                q = q + (ds < (T)0 ? -acc : acc);
                nj = ds < (T)0 ? -nj : nj;
              }
            }
            jumps[b][u * CH + k][v][lane] = nj;
          }
          noise[b][u * CH + k][v][lane] = q;
        }
      }
    }
  };

  // One step of the recursion from the noise q.
  auto advance = [&](int s, const T (&q)[M], const int (&nj)[M]) {
    const T* c = coef + (int64_t)s * a.ncoef;
    const T* p = c + a.poff;
    if constexpr (kHeston) {
      using Lay = HestonLayout<D>;
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int ix = Lay::xi(i), iy = Lay::yi(i);
        heston_next<T>(x[ix], x[iy], cnt[i], p[i], p[N + i], p[2 * N + i], p[3 * N + i],
                       p[4 * N + i], c[0], q[ix], q[iy]);
      }
    } else {
#pragma unroll
      for (int v = 0; v < M; ++v) {
        if constexpr (kCIR)
          x[v] = cir_next<T>(x[v], p[v], p[M + v], p[2 * M + v], c[0], q[v]);
        else if constexpr (kOU)
          x[v] = p[v] * x[v] + q[v];
        else
          x[v] = x[v] + q[v];
        if constexpr (kJump) {
          cnt[v] += nj[v];
          interval_jumps += nj[v];
        }
      }
    }
  };

  // The chunk's output rows, lane k the one reached after its step k (-1:
  // none).  Which steps store, and which of those this wave stores (every W-th
  // row), become scalar masks, so that a step without a store of its own
  // costs no memory wait and groups of such steps no branch.
  static_assert(L <= 64, "one lane per step of a chunk");
  auto rows_of = [&](int c0) -> int {
    return lane < L && c0 + lane < n ? store_row[c0 + lane] : -1;
  };
  int stored = 0;  // rows stored before the chunk
  // K steps from step k0 of the chunk, their LDS and table loads in flight
  // together.
  constexpr int G = M > 2 ? 4 : 8;
  auto steps = [&](int c0, int b, int k0, int rows, uint64_t any, uint64_t mine, auto count) {
    constexpr int K = decltype(count)::value;
    T q[K][M];
    int nj[K][M];
#pragma unroll
    for (int k = 0; k < K; ++k) {
#pragma unroll
      for (int v = 0; v < M; ++v) {
        q[k][v] = noise[b][k0 + k][v][lane];
        nj[k][v] = 0;
        if constexpr (kJump) nj[k][v] = jumps[b][k0 + k][v][lane];
      }
    }
    const uint32_t st = (uint32_t)(any >> k0) & ((1u << K) - 1u);
    const uint32_t my = (uint32_t)(mine >> k0) & ((1u << K) - 1u);
    if ((kJump ? st : my) == 0u) {
#pragma unroll
      for (int k = 0; k < K; ++k) advance(c0 + k0 + k, q[k], nj[k]);
      return;
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      advance(c0 + k0 + k, q[k], nj[k]);
      if ((my >> k) & 1u) {
        const int row = __builtin_amdgcn_readlane(rows, k0 + k);
        store(row);
        if constexpr (kJump) {
          if (a.info_rows) add_interval_jumps(a, row, live, interval_jumps);
        }
      }
      if constexpr (kJump) interval_jumps = (st >> k) & 1u ? 0 : interval_jumps;
    }
  };

  int rows = rows_of(0);
  if (n > 0) draw(0, 0);
  __syncthreads();
  for (int c0 = 0, b = 0; c0 < n; c0 += L, b ^= 1) {
    const int next = rows_of(c0 + L);
    if (c0 + L < n) draw(c0 + L, b ^ 1);
    const uint64_t any = __ballot(rows >= 0);
    const int before = __builtin_amdgcn_mbcnt_hi((uint32_t)(any >> 32),
                                                 __builtin_amdgcn_mbcnt_lo((uint32_t)any, 0));
    const uint64_t mine = __ballot(rows >= 0 && (stored + before) % W == w);
    stored = (stored + __builtin_popcountll(any)) % W;
    const int m = n - c0 < L ? n - c0 : L;
    int k0 = 0;
    for (; k0 + G <= m; k0 += G) steps(c0, b, k0, rows, any, mine, Count<G>{});
    for (; k0 < m; ++k0) steps(c0, b, k0, rows, any, mine, Count<1>{});
    rows = next;
    __syncthreads();
  }

  if (a.info_paths && (kHeston || kJump) && w == 0 && live) {
#pragma unroll
    for (int v = 0; v < N; ++v) a.info_paths[v * P + gid] = cnt[v];
  }
}

template <typename T>
EulerKernel<T> euler_split_kernel(int model, int m, int d, int64_t blocks, bool stream);
template <>
EulerKernel<float> euler_split_kernel<float>(int model, int m, int d, int64_t blocks, bool stream);
template <>
EulerKernel<double> euler_split_kernel<double>(int model, int m, int d, int64_t blocks,
                                               bool stream);

template <int MODEL, typename T, bool STREAM, int MAX, int MOST = 8>
EulerKernel<T> pick_split(int m) {
  if (m == 1) return k_euler_split<MODEL, T, 1, 1, STREAM, MOST>;
  if (m == 2) return k_euler_split<MODEL, T, 2, 1, STREAM, MOST>;
  if constexpr (MAX > 2) {
    if (m == 3) return k_euler_split<MODEL, T, 3, 1, STREAM, MOST>;
    if (m == 4) return k_euler_split<MODEL, T, 4, 1, STREAM, MOST>;
  }
  return nullptr;
}

// Models whose recursion takes a square root.
constexpr bool split_root(int model) {
  return model == SDEGPU_MODEL_CIR || model == SDEGPU_MODEL_HESTON;
}

template <typename T, bool STREAM>
EulerKernel<T> pick_split(int model, int m, int d, int64_t blocks) {
  constexpr bool kRootStream = STREAM || sizeof(T) == 8;
  switch (model) {
    case SDEGPU_MODEL_WIENER: return pick_split<SDEGPU_MODEL_WIENER, T, STREAM, 4>(m);
    case SDEGPU_MODEL_LOGNORM: return pick_split<SDEGPU_MODEL_LOGNORM, T, STREAM, 4>(m);
    case SDEGPU_MODEL_OU: return pick_split<SDEGPU_MODEL_OU, T, STREAM, 4>(m);
    case SDEGPU_MODEL_CIR: return pick_split<SDEGPU_MODEL_CIR, T, kRootStream, 4>(m);
    case SDEGPU_MODEL_JUMPDIFF:
      // (split_waves gives such grids 4 waves a block at most)
      if (sizeof(T) == 8 && blocks > 3 * 256)
        return pick_split<SDEGPU_MODEL_JUMPDIFF, T, STREAM, 2, 4>(m);
      return pick_split<SDEGPU_MODEL_JUMPDIFF, T, STREAM, 2>(m);
    case SDEGPU_MODEL_HESTON:
      if (m == 2) return k_euler_split<SDEGPU_MODEL_HESTON, T, 2, 1, kRootStream>;
      if (m == 4 && d == 1) return k_euler_split<SDEGPU_MODEL_HESTON, T, 4, 1, kRootStream>;
      if (m == 4 && d == 2) return k_euler_split<SDEGPU_MODEL_HESTON, T, 4, 2, kRootStream>;
      return nullptr;
    default: return nullptr;
  }
}

// The kernel for a model, its components m, Heston's group width d, the blocks of the
// grid and rows that begin on 64-byte lines or don't, or null (euler_split_f32.hip,
// euler_split_f64.hip).
#define SDEGPU_EULER_SPLIT_SET(T)                                                         \
  template <>                                                                             \
  EulerKernel<T> euler_split_kernel<T>(int model, int m, int d, int64_t blocks,           \
                                       bool stream) {                                     \
    return stream ? pick_split<T, true>(model, m, d, blocks)                              \
                  : pick_split<T, false>(model, m, d, blocks);                            \
  }

}  // namespace sdegpu
