// Factor and solve of systems with small blocks (n <= 32), one task per node
// and one launch per level: all of a node's work of a level -- the updates it
// receives from the level below, its factor and inverse, its couplings and its
// right-hand sides -- by one (n <= 16) or two (n <= 32) wavefronts.
//
// Level l (s = 2^l, h = s/2), node tasks, k = (2t+1)s - 1:
//   L_k  -= R_{k-h} R_{k-h}^T + Lc_{k+h}^T Lc_{k+h},   the syrk updates,
//   Lc_k  = -R_{k-h} Lc_{k-h},  R_k = -R_{k+h} Lc_{k+h}, the fill-ins
//   y_k  -= R_{k-h} y_{k-h} + Lc_{k+h}^T y_{k+h}         (l > 0), then
//   L_k <- chol(L_k),  R_k <- R_k L_k^-T,  Lc_k <- L_k^-1 Lc_k,
//   y_k <- L_k^-1 y_k;
// target tasks (l > 0), j = 2s(u+1) - 1, the receiving blocks of level l-1 that
// are not nodes of level l: the same updates of L_j and y_j.
// (syrk, gemm, potrf, trsm and forward sweep of block_tridiag_solver.py:797-813
// and :425-485; fill-ins never go to memory before they are couplings.)
// A task reads only blocks finished at an earlier level and writes its own, so
// a level needs no atomics and results are bitwise reproducible.
// Backward, per node: x_k <- L_k^-T (x_k - R_k^T x_{k+s} - Lc_k x_{k-s}).
//
// How a node task works:
// * Updates on MFMA with operands straight from global memory in the operand
//   layout (no LDS): in R R^T and Lc^T Lc both operands are the same registers.
// * The factor runs as 16-column panels (nd_panel.h).  Everything that needs
//   L^-T from the right is a payload row: the identity (the transposed
//   inverse), rows of R_k, columns of Lc_k, columns of y_k.  n <= 16: these are
//   exactly the 64 lanes of one wavefront.  n <= 32: wavefront 0 takes the
//   identity, the lower rows of L_k and the right-hand sides, wavefront 1 R_k
//   and Lc_k; both factor the 16x16 diagonal tile, which costs less than
//   handing its columns over.  Between the panels one MFMA update per tile.
//
// What bounds it.  Wide levels: HBM (256 systems of n=32 N=128 m=4 FP64: level 0
// moves 805 MB in 176 us, 4.6 TB/s; all factor levels 570 us, backward 209 us).
// Narrow levels: one task's latency and its launch, 9-10 us at n=32, 4.7 us at
// n=12, 4 and 2.5 us backward.  It replaces separate factor, trsm, Schur and
// sweep launches (FP64 factor_and_solve n=12 N=20 126 -> 35 us, n=32 N=100 136 ->
// 96 us, 256 systems of n=20 N=61 FP32 345 -> 157 us).  Blocks are read with
// 32-bit offsets from a scalar base and no branch per element: with generic
// pointers and selected loads the n=20 FP32 task took 17 us instead of 6.
#include <algorithm>
#include <new>
#include <stdexcept>
#include <vector>

#include "../../include/socu_hip.h"
#include "nd_common.h"
#include "nd_internal.h"
#include "nd_small.h"
#include "nd_tile.h"

namespace socu {

namespace {

// Kernel variants: K4 = ceil(n / 4).  n <= 16 NB, the last of the NB 16-column
// panels has NC columns, and products sum over 4 K4 entries.  EX: n == 4 K4
// (every index a compile-time constant, no masks).
template <typename T, int K4, bool EX>
struct SmallShape {
  static constexpr int NB = (K4 + 3) / 4;
  static constexpr int NC = 4 * K4 - 16 * (NB - 1);
  static constexpr int NP = 16 * NB;
  static constexpr int P = NP + 1;
  static constexpr int kZ = 32;                 // 31 entries: rows of the identity
  static constexpr int kTile = NP * P;
  static constexpr int kFixed = 3 * kTile + kZ;  // L_k, R_k, Lc_k^T, identity
  static __host__ __device__ constexpr int elems(int m) { return kFixed + m * P; }
};

// MFMA operands of an n x n block: [t][b] holds rows 16b + lane % 16 at
// column 4t + lane / 16 (ROW), or the transpose: columns 16b + lane % 16 at row
// 4t + lane / 16.  Rows and columns past n repeat the last one: such rows of a
// product are never used.  mask_k: zeros past n in the summed direction
// (one of a product's two operands needs them).
template <typename T, int K4, bool EX, bool ROW>
struct Frag {
  static constexpr int NB = (K4 + 3) / 4;
  T f[K4][NB];
  __device__ __forceinline__ void load(const T* M, int n) {
    const int l = lane_id(), i = l & 15, g = l >> 4;
    int o[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int r = EX ? 16 * b + i : min(16 * b + i, n - 1);
      o[b] = (EX && 16 * b + 16 > 4 * K4) ? min(r, 4 * K4 - 1) : r;
      if (ROW) o[b] *= n;
    }
#pragma unroll
    for (int t = 0; t < K4; ++t) {
      const int k = EX ? 4 * t + g : min(4 * t + g, n - 1);
#pragma unroll
      for (int b = 0; b < NB; ++b) f[t][b] = ldg(M, ROW ? o[b] + k : k * n + o[b]);
    }
  }
  __device__ __forceinline__ void mask_k(int n) {
    if constexpr (!EX) {
      // (the smallest variant of two wavefronts also takes n <= 16, with
      // m > 16)
      const int g = lane_id() >> 4;
#pragma unroll
      for (int t = K4 == 5 ? 0 : K4 - 1; t < K4; ++t)
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          pin_reg(f[t][b]);
          f[t][b] = (4 * t + g < n) ? f[t][b] : T(0);
        }
    }
  }
};

// Right-hand sides, columns c0 .. c0 + 15: as the MFMA B operand ([t]: row
// 4t + lane / 16) and in the accumulators' layout.  Entries past n or m repeat
// others; the first operand is masked in the summed direction and results
// past n or m are not stored.  FAR: block rows of any size (the factor takes m <= 32).
template <typename T, int K4, bool FAR = false>
__device__ __forceinline__ void ld_rhs_b(T (&f)[K4], const T* y, int n, int m, int c0) {
  const int l = lane_id(), j = min(c0 + (l & 15), m - 1), g = l >> 4;
#pragma unroll
  for (int t = 0; t < K4; ++t) f[t] = ld_rhs<FAR>(y, min(4 * t + g, n - 1), m, j);
}
template <typename T, int NB, bool FAR = false>
__device__ __forceinline__ void ld_rhs_acc(typename Mfma<T>::acc_t (&a)[NB], const T* y, int n, int m, int c0) {
  const int l = lane_id(), j = min(c0 + (l & 15), m - 1);
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 4; ++r) a[b][r] = ld_rhs<FAR>(y, min(16 * b + Mfma<T>::row(l, r), n - 1), m, j);
}
// acc += A B (tiles i, j of A's and B's rows; LOWER: j <= i only).
template <typename T, int K4, bool EX, bool RA, bool RB, bool LOWER, int NT>
__device__ __forceinline__ void mma_frags(typename Mfma<T>::acc_t (&acc)[NT], const Frag<T, K4, EX, RA>& A,
                                          const Frag<T, K4, EX, RB>& B) {
  constexpr int NB = (K4 + 3) / 4;
#pragma unroll
  for (int t = 0; t < K4; ++t)
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int j = 0; j < (LOWER ? i + 1 : NB); ++j) {
        const int q = LOWER ? i * (i + 1) / 2 + j : i * NB + j;
        acc[q] = Mfma<T>::mma(A.f[t][i], B.f[t][j], acc[q]);
      }
}
template <typename T, int K4, bool EX, bool RA>
__device__ __forceinline__ void mma_rhs(typename Mfma<T>::acc_t (&acc)[(K4 + 3) / 4], const Frag<T, K4, EX, RA>& A,
                                        const T (&y)[K4]) {
#pragma unroll
  for (int t = 0; t < K4; ++t)
#pragma unroll
    for (int i = 0; i < (K4 + 3) / 4; ++i) acc[i] = Mfma<T>::mma(A.f[t][i], y[t], acc[i]);
}

// What a block row j receives from level l-1: its diagonal block's lower tiles
// (accumulator layout, tile (i, b) at i (i + 1) / 2 + b) and its right-hand
// sides.  Ra, Lcc: NULL where there is none.
template <typename T, int K4, bool EX>
struct Pull {
  static constexpr int NB = (K4 + 3) / 4, NTRI = NB * (NB + 1) / 2;
  typename Mfma<T>::acc_t d[NTRI];  // L_j
  typename Mfma<T>::acc_t y[NB];    // columns c0 .. of y_j
  Frag<T, K4, EX, true> fr;
  Frag<T, K4, EX, false> fc;

  __device__ __forceinline__ void run(const T* Lin, const T* Ra, const T* Lcc, const T* yj, const T* ya, const T* yc,
                                      int n, int m) {
    const int l = lane_id();
    T va[K4], vc[K4];
    if (Ra != nullptr) fr.load(Ra, n);
    if (Lcc != nullptr) fc.load(Lcc, n);
    if (yj != nullptr) {
      ld_rhs_acc<T, NB>(y, yj, n, m, 0);
      if (Ra != nullptr) ld_rhs_b<T, K4>(va, ya, n, m, 0);
      if (Lcc != nullptr) ld_rhs_b<T, K4>(vc, yc, n, m, 0);
    }
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int b = 0; b <= i; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int row = 16 * i + Mfma<T>::row(l, e), col = 16 * b + (l & 15);
          d[i * (i + 1) / 2 + b][e] = ldg(Lin, min(row, n - 1) * n + min(col, n - 1));
        }
    if (Ra != nullptr) fr.mask_k(n);
    if (Lcc != nullptr) fc.mask_k(n);
    if (Ra != nullptr || Lcc != nullptr) {
      typename Mfma<T>::acc_t u[NTRI];
#pragma unroll
      for (int q = 0; q < NTRI; ++q) u[q] = acc_zero<T>();
      if (Ra != nullptr) {
        mma_frags<T, K4, EX, true, true, true>(u, fr, fr);
        mfma_settle<T>();
      }
      if (Lcc != nullptr) {
        mma_frags<T, K4, EX, false, false, true>(u, fc, fc);
        mfma_settle<T>();
      }
#pragma unroll
      for (int q = 0; q < NTRI; ++q) d[q] -= u[q];
    }
    if (yj != nullptr) sub_rhs(Ra != nullptr, Lcc != nullptr, va, vc);
  }
  __device__ __forceinline__ void sub_rhs(bool ra, bool lc, const T (&va)[K4], const T (&vc)[K4]) {
    if (!ra && !lc) return;
    typename Mfma<T>::acc_t u[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) u[i] = acc_zero<T>();
    if (ra) {
      mma_rhs<T, K4, EX, true>(u, fr, va);
      mfma_settle<T>();
    }
    if (lc) {
      mma_rhs<T, K4, EX, false>(u, fc, vc);
      mfma_settle<T>();
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) y[i] -= u[i];
  }
  // the next 16 columns of y_j (the operands are still in registers)
  __device__ __forceinline__ void more_rhs(bool ra, bool lc, const T* yj, const T* ya, const T* yc, int n, int m,
                                           int c0) {
    T va[K4], vc[K4];
    ld_rhs_acc<T, NB>(y, yj, n, m, c0);
    if (ra) ld_rhs_b<T, K4>(va, ya, n, m, c0);
    if (lc) ld_rhs_b<T, K4>(vc, yc, n, m, c0);
    sub_rhs(ra, lc, va, vc);
  }
};

// -A B of two n x n blocks into LDS: Q[r][c], or Q[c][r] (TR).
template <typename T, int K4, bool EX, bool TR>
__device__ __forceinline__ void fill_in(T* Q, const T* A, const T* B, int n) {
  using Sh = SmallShape<T, K4, EX>;
  constexpr int NB = Sh::NB, P = Sh::P;
  typename Mfma<T>::acc_t acc[NB * NB];
  Frag<T, K4, EX, true> fa;
  Frag<T, K4, EX, false> fb;
  fa.load(A, n);
  fb.load(B, n);
#pragma unroll
  for (int q = 0; q < NB * NB; ++q) acc[q] = acc_zero<T>();
  fa.mask_k(n);
  mma_frags<T, K4, EX, true, false, false>(acc, fa, fb);
  const int l = lane_id();
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * i + Mfma<T>::row(l, r), col = 16 * j + (l & 15);
        Q[TR ? col * P + row : row * P + col] = -acc[i * NB + j][r];
      }
}

// An n x n block into LDS and back: Q[r][c], or Q[c][r] (TR).  (Rows and
// columns past n repeat the last ones: payload rows and entries past n are
// never used.)
template <typename T, int K4, bool EX, bool TR>
__device__ __forceinline__ void copy_in(T* Q, const T* M, int n) {
  using Sh = SmallShape<T, K4, EX>;
  constexpr int P = Sh::P, RP = 64 / Sh::NP;  // rows per step
  const int l = lane_id(), lr = l / Sh::NP, lc = l % Sh::NP;
  T v[4 * K4 / RP];
#pragma unroll
  for (int q = 0; q < 4 * K4 / RP; ++q) v[q] = ldg(M, min(RP * q + lr, n - 1) * n + min(lc, n - 1));
#pragma unroll
  for (int q = 0; q < 4 * K4 / RP; ++q) {
    const int r = RP * q + lr;
    Q[TR ? lc * P + r : r * P + lc] = v[q];
  }
}
template <typename T, int K4, bool EX, bool TR>
__device__ __forceinline__ void copy_out(T* M, const T* Q, int n) {
  using Sh = SmallShape<T, K4, EX>;
  constexpr int P = Sh::P, RP = 64 / Sh::NP;
  const int l = lane_id(), lr = l / Sh::NP, lc = l % Sh::NP;
  T v[4 * K4 / RP];
#pragma unroll
  for (int q = 0; q < 4 * K4 / RP; ++q) {
    const int r = RP * q + lr;
    v[q] = Q[TR ? lc * P + r : r * P + lc];
  }
  if (lc < n) {
#pragma unroll
    for (int q = 0; q < 4 * K4 / RP; ++q)
      if (EX || RP * q + lr < n) stg(M, (RP * q + lr) * n + lc, v[q]);
  }
}

template <typename T, int NB>
__device__ __forceinline__ void rhs_to_lds(T* Y, typename Mfma<T>::acc_t (&a)[NB], int m, int c0) {
  constexpr int P = 16 * NB + 1;
  const int l = lane_id(), j = c0 + (l & 15);
  if (j < m)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) Y[j * P + 16 * b + Mfma<T>::row(l, r)] = a[b][r];
}

// Second half of 16 rows Q (pitch P) -= X L21^T, X being their first half; b:
// L21 as the B operand.  rows: how many exist (reads are clamped, writes
// masked).
template <typename T>
__device__ __forceinline__ void half_update(T* Q, int P, const T (&b)[4], int rows) {
  const int l = lane_id(), i = min(l & 15, rows - 1), g = l >> 4;
  typename Mfma<T>::acc_t acc;
#pragma unroll
  for (int r = 0; r < 4; ++r) acc[r] = Q[min(Mfma<T>::row(l, r), rows - 1) * P + 16 + (l & 15)];
  T a[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) a[t] = Q[i * P + 4 * t + g];
#pragma unroll
  for (int t = 0; t < 4; ++t) acc = Mfma<T>::mma(-a[t], b[t], acc);
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (Mfma<T>::row(l, r) < rows) Q[Mfma<T>::row(l, r) * P + 16 + (l & 15)] = acc[r];
}

// One node or target task of level l by the NB wavefronts of a task slot
// (w: this wavefront's number in it).  task < dim: node; else the pair of
// targets NB (task - dim) .. (one per wavefront).  `run` is uniform over the
// slot; every wavefront of the workgroup reaches the barriers (n > 16 only).
template <typename T, int K4, bool EX>
__device__ __forceinline__ void up_task(const SmallSys<T>& Q, int l, int task, bool run, T* lds, int w) {
  using Sh = SmallShape<T, K4, EX>;
  constexpr int P = Sh::P, NB = Sh::NB, NC = Sh::NC;
  const int N = Q.N, n = EX ? 4 * K4 : Q.n, m = Q.m;
  const int nn = n * n, nm = n * m;
  const int s = 1 << l, h = s >> 1;
  const int dim = (N + s) / (2 * s);
  const int lane = lane_id(), r = lane & 15, g = lane >> 4;
  const int offp = seg_offset(N, l > 0 ? l - 1 : 0);
  const int off = l > 0 ? offp + (N >> (l - 1)) - 1 : 0;
  T* const S = lds;
  T* const PR = S + Sh::kTile;
  T* const PC = PR + Sh::kTile;
  T* const Z = PC + Sh::kTile;
  T* const Y = Z + Sh::kZ;
  const bool node = run && task < dim;
  // L is first read at level 0 (its nodes) and level 1 (everything else)
  const T* const Lin = l <= 1 ? Q.Lin : Q.L;
  // block row of a node task; a target task's depends on the wavefront
  const int k = node ? s - 1 + 2 * s * task : 2 * s * (NB * (task - dim) + w + 1) - 1;
  const bool hasR = node && k + s < N, hasC = node && k >= s;
  T* const Rk = Q.E + (size_t)(off + (k >> l)) * nn;
  T* const Lck = Q.E + (size_t)(off + ((k - s) >> l)) * nn;
  T* const yk = Q.x != nullptr ? Q.x + (size_t)k * nm : nullptr;
  const T* Ra = l > 0 ? Q.E + (size_t)(offp + ((k - h) >> (l - 1))) * nn : nullptr;          // (k, k-h)
  const T* Lcc = l > 0 && k + h < N ? Q.E + (size_t)(offp + (k >> (l - 1))) * nn : nullptr;  // (k+h, k)

  if (run && (node ? w == 0 : k < N)) {
    Pull<T, K4, EX> pull;
    pull.run(Lin + (size_t)k * nn, Ra, Lcc, yk, yk - (size_t)h * nm, yk + (size_t)h * nm, n, m);
    if (node) {
      if (lane < Sh::kZ) Z[lane] = lane == 15 ? T(1) : T(0);
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j <= i; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int row = 16 * i + Mfma<T>::row(lane, e), col = 16 * j + r;
            T v = pull.d[i * (i + 1) / 2 + j][e];
            if (!(EX && 4 * K4 >= 16 * i + 16))  // identity padding
              v = (row < n && col < n) ? v : ((row == col) ? T(1) : T(0));
            S[row * P + col] = v;
          }
    } else {
      T* Lj = Q.L + (size_t)k * nn;
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j <= i; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int row = 16 * i + Mfma<T>::row(lane, e), col = 16 * j + r;
            if (col <= row && row < n) stg(Lj, row * n + col, pull.d[i * (i + 1) / 2 + j][e]);
          }
    }
    if (yk != nullptr)
      for (int c0 = 0; c0 < m; c0 += 16) {
        if (c0 > 0)
          pull.more_rhs(Ra != nullptr, Lcc != nullptr, yk, yk - (size_t)h * nm, yk + (size_t)h * nm, n, m, c0);
        if (node) {
          rhs_to_lds<T, NB>(Y, pull.y, m, c0);
        } else if (c0 + r < m) {
#pragma unroll
          for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int row = 16 * b + Mfma<T>::row(lane, e);
              if (row < n) stg(yk, row * m + c0 + r, pull.y[b][e]);
            }
        }
      }
  }
  if (node && w == NB - 1) {
    if (l == 0) {
      if (hasR) copy_in<T, K4, EX, false>(PR, Q.Ein + (Rk - Q.E), n);
      if (hasC) copy_in<T, K4, EX, true>(PC, Q.Ein + (Lck - Q.E), n);
    } else {
      // R_{k+h} Lc_{k+h} and R_{k-h} Lc_{k-h}
      if (hasR) fill_in<T, K4, EX, false>(PR, Q.E + (size_t)(offp + ((k + h) >> (l - 1))) * nn, Lcc, n);
      if (hasC) fill_in<T, K4, EX, true>(PC, Ra, Q.E + (size_t)(offp + ((k - s) >> (l - 1))) * nn, n);
    }
  }

  if constexpr (NB == 1) {
    if (!node) return;
    wave_lds_order();
    T u[16], p[1][16];
    // payload rows: identity, R_k, Lc_k^T, y_k^T
    const bool has = g == 0 || (g == 1 && hasR) || (g == 2 && hasC) || (g == 3 && yk != nullptr && r < m);
    T* row = g == 1 ? PR + r * P : (g == 2 ? PC + r * P : Y + r * P);
    run_panel<T, 1, NC>(u, p, S + r * P, (g == 0 || !has) ? Z + 15 - r : row);
    if (g == 0) row = S + r * P;
    const int rl = g == 0 ? r : -1;
    if (has) {
#pragma unroll
      for (int c = 0; c < NC; ++c) row[c] = (c <= rl) ? u[c] : p[0][c];
    }
    wave_lds_order();
    copy_out<T, K4, EX, false>(Q.L + (size_t)k * nn, S, n);
    if (hasR) copy_out<T, K4, EX, false>(Rk, PR, n);
    if (hasC) copy_out<T, K4, EX, true>(Lck, PC, n);
    if (yk != nullptr)
      for (int idx = lane; idx < 16 * m; idx += 64) {
        const int j = idx >> 4, i = idx & 15;
        if (i < n) stg(yk, i * m + j, Y[j * P + i]);
      }
    return;
  } else {
    __syncthreads();
    T u[16], p[1][16];
    // payload rows of wavefront 0: identity (lanes 0-15), the lower rows of
    // L_k (16-31), y_k^T (32-63); of wavefront 1: R_k (0-31), Lc_k^T (32-63)
    const int j32 = lane - 32;
    bool has;
    T* row;
    if (w == 0) {
      row = g == 0 ? S + r * P + 16 : (g == 1 ? S + (16 + r) * P : Y + j32 * P);
      has = g < 2 || (yk != nullptr && j32 < m);
    } else {
      row = lane < 32 ? PR + lane * P : PC + j32 * P;
      has = lane < 32 ? hasR : hasC;
    }
    const T* const ident = Z + 15 - r;
    if (node) {
      run_panel<T, 1, 16>(u, p, S + r * P, (w == 0 && g == 0) || !has ? ident : row);
      if (has) {
#pragma unroll
        for (int c = 0; c < 16; ++c) row[c] = p[0][c];
      }
    }
    __syncthreads();
    if (node) {
      if (w == 0 && g == 0) {  // L_11 with U_11 above its diagonal
#pragma unroll
        for (int c = 0; c < 16; ++c) S[r * P + c] = (c <= r) ? u[c] : p[0][c];
      }
      T b[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) b[t] = S[(16 + r) * P + 4 * t + g];
      if (w == 0) {
        // U_12 = -U_11 L_21^T (U_11 parked in the tile that receives it)
        typename Mfma<T>::acc_t s22, u12 = acc_zero<T>();
        T a[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) a[t] = S[r * P + 16 + 4 * t + g];
#pragma unroll
        for (int e = 0; e < 4; ++e) s22[e] = S[(16 + Mfma<T>::row(lane, e)) * P + 16 + r];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          s22 = Mfma<T>::mma(-b[t], b[t], s22);
          u12 = Mfma<T>::mma(-a[t], b[t], u12);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          S[(16 + Mfma<T>::row(lane, e)) * P + 16 + r] = s22[e];
          S[Mfma<T>::row(lane, e) * P + 16 + r] = u12[e];
        }
        if (yk != nullptr)
          for (int c0 = 0; c0 < m; c0 += 16) half_update<T>(Y + c0 * P, P, b, min(16, m - c0));
      } else {
        if (hasR) {
          half_update<T>(PR, P, b, 16);
          half_update<T>(PR + 16 * P, P, b, 16);
        }
        if (hasC) {
          half_update<T>(PC, P, b, 16);
          half_update<T>(PC + 16 * P, P, b, 16);
        }
      }
    }
    __syncthreads();
    if (node) {
      // (lanes 16-31 of wavefront 0: the identity rows of the second tile)
      const bool id = w == 0 && g == 1;
      T* row2 = row + 16;
      if (w == 0 && g == 0) row2 = row;  // U_12
      run_panel<T, 1, NC>(u, p, S + (16 + r) * P + 16, id || !has ? ident : row2);
      if (has && !id) {
#pragma unroll
        for (int c = 0; c < NC; ++c) row2[c] = p[0][c];
      }
    }
    __syncthreads();
    if (!node) return;
    if (w == 0) {
      if (g == 1) {
#pragma unroll
        for (int c = 0; c < NC; ++c) S[(16 + r) * P + 16 + c] = (c <= r) ? u[c] : p[0][c];
      }
      wave_lds_order();
      copy_out<T, K4, EX, false>(Q.L + (size_t)k * nn, S, n);
      if (yk != nullptr)
        for (int idx = lane; idx < 32 * m; idx += 64) {
          const int j = idx >> 5, i = idx & 31;
          if (i < n) stg(yk, i * m + j, Y[j * P + i]);
        }
    } else {
      if (hasR) copy_out<T, K4, EX, false>(Rk, PR, n);
      if (hasC) copy_out<T, K4, EX, true>(Lck, PC, n);
    }
  }
}

// One block row's forward step of level l by one wavefront (columns c0 ..
// c1 - 1 of the right-hand sides): with upd it receives from level l-1 (nodes
// of level l, then the other targets of level l-1), with app nodes apply
// y_k <- L_k^-1 y_k, from the inverse stored above the diagonal.
template <typename T, int K4, bool EX, bool FAR>
__device__ __forceinline__ void forward_task(const SmallSys<T>& Q, int l, int task, bool upd, bool app, int c0,
                                             int c1) {
  constexpr int NB = (K4 + 3) / 4;
  constexpr int KU = sizeof(T) == 8 ? K4 : 4 * NB;
  const int N = Q.N, n = EX ? 4 * K4 : Q.n, m = Q.m;
  const int nn = n * n;
  const std::conditional_t<FAR, size_t, int> nm = (decltype(nm))n * m;
  const int s = 1 << l, h = s >> 1, dim = (N + s) / (2 * s);
  const bool node = task < dim;
  app = app && node;
  upd = upd && l > 0;
  const int k = node ? s - 1 + 2 * s * task : 2 * s * (task - dim + 1) - 1;
  const int offp = seg_offset(N, l > 0 ? l - 1 : 0);
  const T* Ra = upd ? Q.E + (size_t)(offp + ((k - h) >> (l - 1))) * nn : nullptr;          // (k, k-h)
  const T* Lcc = upd && k + h < N ? Q.E + (size_t)(offp + (k >> (l - 1))) * nn : nullptr;  // (k+h, k)
  const T* Lk = Q.L + (size_t)k * nn;
  T* yk = Q.x + (size_t)k * nm;
  const int lane = lane_id(), i = lane & 15;
  Frag<T, K4, EX, true> fr;
  Frag<T, K4, EX, false> fc;
  T y[K4], y2[K4];
  typename Mfma<T>::acc_t a[NB];
  if (upd) {
    fr.load(Ra, n);
    ld_rhs_b<T, K4, FAR>(y, yk - (size_t)h * nm, n, m, c0);
  }
  if (Lcc != nullptr) {
    fc.load(Lcc, n);
    ld_rhs_b<T, K4, FAR>(y2, yk + (size_t)h * nm, n, m, c0);
  }
  ld_rhs_acc<T, NB, FAR>(a, yk, n, m, c0);
  // L_k^-1, rows 16b + i, from the tiles on and above the stored diagonal
  T fu[KU][NB], dg[NB];
  if (app) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int row = min(16 * b + i, n - 1);
      dg[b] = ldg(Lk, row * (n + 1));
#pragma unroll
      for (int t = 0; t < min(KU, 4 * b + 4); ++t) {
        const int kr = 16 * (t / 4) + Mfma<T>::row(lane, t % 4);
        fu[t][b] = ldg(Lk, min(kr, n - 1) * n + row);
      }
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      pin_reg(dg[b]);
      dg[b] = T(1) / dg[b];
#pragma unroll
      for (int t = 4 * b; t < min(KU, 4 * b + 4); ++t) {
        const int kr = 16 * b + Mfma<T>::row(lane, t % 4), row = 16 * b + i;
        pin_reg(fu[t][b]);
        fu[t][b] = (kr < row) ? fu[t][b] : ((kr == row) ? dg[b] : T(0));
      }
    }
  }
  if (upd) fr.mask_k(n);
  if (Lcc != nullptr) fc.mask_k(n);
  for (const int first = c0; c0 < c1; c0 += 16) {
    if (c0 > first) {
      if (upd) ld_rhs_b<T, K4, FAR>(y, yk - (size_t)h * nm, n, m, c0);
      if (Lcc != nullptr) ld_rhs_b<T, K4, FAR>(y2, yk + (size_t)h * nm, n, m, c0);
      ld_rhs_acc<T, NB, FAR>(a, yk, n, m, c0);
    }
    typename Mfma<T>::acc_t u[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) u[b] = acc_zero<T>();
    if (upd) {
      mma_rhs<T, K4, EX, true>(u, fr, y);
      mfma_settle<T>();
    }
    if (Lcc != nullptr) {
      mma_rhs<T, K4, EX, false>(u, fc, y2);
      mfma_settle<T>();
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) a[b] -= u[b];
    if (app) {
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        u[b] = acc_zero<T>();
#pragma unroll
        for (int t = 0; t < min(KU, 4 * b + 4); ++t) u[b] = Mfma<T>::mma(fu[t][b], a[t / 4][t % 4], u[b]);
      }
      mfma_settle<T>();
#pragma unroll
      for (int b = 0; b < NB; ++b) a[b] = u[b];
    }
    if (c0 + i < m)
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int row = 16 * b + Mfma<T>::row(lane, e);
          if (row < n) st_rhs<FAR>(yk, row, m, c0 + i, a[b][e]);
        }
  }
}

// x_k <- U (x_k - R_k^T x_{k+s} - Lc_k x_{k-s}) with U = L_k^-T as stored, by
// one wavefront (columns c0 .. c1 - 1): three products on MFMA, operands from global memory.  The
// right-hand sides are the (up to 16) columns of the B operand; the difference
// goes from the accumulators to the second product's B operand as it is: row
// kr(t) of lane group g below is the row an accumulator's entry t holds.
template <typename T, int K4, bool EX, bool FAR>
__device__ __forceinline__ void down_task(const SmallSys<T>& Q, int l, int t0, int c0, int c1) {
  constexpr int NB = (K4 + 3) / 4;
  // steps of the second product (FP32: an accumulator's entry t spans the
  // whole 16-row tile)
  constexpr int KU = sizeof(T) == 8 ? K4 : 4 * NB;
  const int N = Q.N, n = EX ? 4 * K4 : Q.n, m = Q.m;
  const int nn = n * n;
  const std::conditional_t<FAR, size_t, int> nm = (decltype(nm))n * m;
  const int s = 1 << l, k = s - 1 + 2 * s * t0;
  const int off = seg_offset(N, l);
  const bool hasR = k + s < N, hasC = k >= s;
  const T* Rk = Q.E + (size_t)(off + (k >> l)) * nn;
  const T* Lck = Q.E + (size_t)(off + ((k - s) >> l)) * nn;
  const T* Lk = Q.L + (size_t)k * nn;
  T* xk = Q.x + (size_t)k * nm;
  const int lane = lane_id(), i = lane & 15;
  Frag<T, K4, EX, false> fr;
  Frag<T, K4, EX, true> fc;
  T y[K4], y2[K4];
  typename Mfma<T>::acc_t a[NB];
  if (hasR) {
    fr.load(Rk, n);
    ld_rhs_b<T, K4, FAR>(y, xk + (size_t)s * nm, n, m, c0);
  }
  if (hasC) {
    fc.load(Lck, n);
    ld_rhs_b<T, K4, FAR>(y2, xk - (size_t)s * nm, n, m, c0);
  }
  ld_rhs_acc<T, NB, FAR>(a, xk, n, m, c0);
  // U[16b + i][kr]: rows of the stored block above its diagonal (tiles on and
  // above it), and the diagonal
  T fu[KU][NB], dg[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int row = 16 * b + i;
    dg[b] = ldg(Lk, min(row, n - 1) * (n + 1));
#pragma unroll
    for (int t = 4 * b; t < KU; ++t) {
      const int kr = 16 * (t / 4) + Mfma<T>::row(lane, t % 4);
      fu[t][b] = ldg(Lk, min(row, n - 1) * n + min(kr, n - 1));
    }
  }
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int row = 16 * b + i;
    pin_reg(dg[b]);
    dg[b] = T(1) / dg[b];
#pragma unroll
    for (int t = 4 * b; t < KU; ++t) {
      const int kr = 16 * (t / 4) + Mfma<T>::row(lane, t % 4);
      pin_reg(fu[t][b]);
      if (t < 4 * b + 4) fu[t][b] = (kr > row) ? fu[t][b] : ((kr == row) ? dg[b] : T(0));
      if (!EX || 16 * (t / 4) + 16 > 4 * K4) fu[t][b] = (kr < n) ? fu[t][b] : T(0);
    }
  }
  if (hasR) fr.mask_k(n);
  if (hasC) fc.mask_k(n);
  for (const int first = c0; c0 < c1; c0 += 16) {
    if (c0 > first) {
      if (hasR) ld_rhs_b<T, K4, FAR>(y, xk + (size_t)s * nm, n, m, c0);
      if (hasC) ld_rhs_b<T, K4, FAR>(y2, xk - (size_t)s * nm, n, m, c0);
      ld_rhs_acc<T, NB, FAR>(a, xk, n, m, c0);
    }
    typename Mfma<T>::acc_t u[NB], o[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) u[b] = o[b] = acc_zero<T>();
    if (hasR) {
      mma_rhs<T, K4, EX, false>(u, fr, y);
      mfma_settle<T>();
    }
    if (hasC) {
      mma_rhs<T, K4, EX, true>(u, fc, y2);
      mfma_settle<T>();
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) a[b] -= u[b];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int t = 4 * b; t < KU; ++t) o[b] = Mfma<T>::mma(fu[t][b], a[t / 4][t % 4], o[b]);
    if (c0 + i < m)
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int row = 16 * b + Mfma<T>::row(lane, e);
          if (row < n) st_rhs<FAR>(xk, row, m, c0 + i, o[b][e]);
        }
  }
}

template <typename T, int K4, bool EX>
__global__ __launch_bounds__(64 * ((K4 + 3) / 4)) void k_small_up(SmallArgs<T> A, int l) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  SmallSys<T> Q;
  int task;
  if (!small_sys(A, Q, task)) return;
  up_task<T, K4, EX>(Q, l, task, true, reinterpret_cast<T*>(smem_raw), wave_uniform());
}

template <typename T, int K4, bool EX, bool FAR>
__global__ __launch_bounds__(64) void k_small_down(SmallArgs<T> A, int l) {
  SmallSys<T> Q;
  int task;
  if (!small_sys(A, Q, task)) return;
  // (grid z: 16 right-hand sides each, or one for all of them)
  const int c0 = 16 * blockIdx.z;
  down_task<T, K4, EX, FAR>(Q, l, task, c0, gridDim.z > 1 ? c0 + 16 : Q.m);
}

template <typename T, int K4, bool EX, bool FAR>
__global__ __launch_bounds__(64) void k_small_forward(SmallArgs<T> A, int l, int upd, int app) {
  SmallSys<T> Q;
  int task;
  if (!small_sys(A, Q, task)) return;
  const int c0 = 16 * blockIdx.z;
  forward_task<T, K4, EX, FAR>(Q, l, task, upd != 0, app != 0, c0, gridDim.z > 1 ? c0 + 16 : Q.m);
}

// Levels lo .. of one system, up and (with right-hand sides) down again, by
// one workgroup, a task per wavefront (n <= 16): the narrow levels, where a
// launch per level and direction costs more than the level, and whole small
// systems.
constexpr int kTailWaves = 16;
constexpr int kTailMaxSystems = 256;

template <typename T, int K4, bool EX>
__global__ __launch_bounds__(64 * kTailWaves) void k_small_tail(SmallArgs<T> A, int lo) {
  using Sh = SmallShape<T, K4, EX>;
  static_assert(Sh::NB == 1, "one wavefront per task");
  extern __shared__ __align__(16) unsigned char smem_raw[];
  SmallSys<T> Q;
  int task;
  if (!small_sys(A, Q, task)) return;
  const int wv = wave_uniform();
  T* lds = reinterpret_cast<T*>(smem_raw) + wv * Sh::elems(A.m);
  const int Lv = recursive_iterations(Q.N);
  for (int l = lo; l < Lv; ++l) {
    const int s = 1 << l, count = (Q.N + s) / (2 * s) + (l > 0 ? Q.N / (2 * s) : 0);
    for (int t = wv; t < count; t += kTailWaves) up_task<T, K4, EX>(Q, l, t, true, lds, 0);
    __syncthreads();
  }
  if (Q.x == nullptr) return;
  for (int l = Lv - 1; l >= lo; --l) {
    const int s = 1 << l, dim = (Q.N + s) / (2 * s);
    for (int t = wv; t < dim; t += kTailWaves) down_task<T, K4, EX, false>(Q, l, t, 0, Q.m);
    __syncthreads();
  }
}

// f(K4, EX as integral constants) for a variant of small_class().
template <int K4 = 1, typename F>
void with_class(int cls, F f) {
  if constexpr (K4 <= kSmallN / 4) {
    if (cls / 2 != K4 - 1) return with_class<K4 + 1>(cls, f);
    if (cls % 2) return f(std::integral_constant<int, K4>{}, std::integral_constant<bool, true>{});
    return f(std::integral_constant<int, K4>{}, std::integral_constant<bool, false>{});
  }
}

template <typename T>
hipError_t set_small_attrs() {
  hipError_t e = hipSuccess;
  for (int cls = 0; cls < kSmallClasses && e == hipSuccess; ++cls)
    with_class(cls, [&](auto k4, auto ex) {
      constexpr int K4 = decltype(k4)::value;
      constexpr bool EX = decltype(ex)::value;
      if constexpr (K4 <= 4)
        e = hipFuncSetAttribute((const void*)k_small_tail<T, K4, EX>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)(sizeof(T) * kTailWaves * SmallShape<T, K4, EX>::elems(16)));
    });
  return e;
}

template <typename T>
void launch_up(int cls, dim3 grid, const SmallArgs<T>& A, int l, hipStream_t st) {
  with_class(cls, [&](auto k4, auto ex) {
    constexpr int K4 = decltype(k4)::value;
    constexpr bool EX = decltype(ex)::value;
    using Sh = SmallShape<T, K4, EX>;
    const size_t lds = sizeof(T) * Sh::elems(A.m);
    hipLaunchKernelGGL((k_small_up<T, K4, EX>), grid, dim3(64 * Sh::NB), lds, st, A, l);
  });
}
// Block rows of right-hand sides of 4 GiB and more take 64-bit offsets, in a variant
// of their own (every n by its padded form): in the common one they cost 1.5% (256
// systems of n=20 N=61 m=1, FP32 factor_and_solve, 157.8 / 160.2 us).
template <typename T>
void launch_down(int cls, dim3 grid, const SmallArgs<T>& A, int l, hipStream_t st) {
  if (far_rhs<T>(A.n, A.m))
    return with_class(cls & ~1, [&](auto k4, auto) {
      hipLaunchKernelGGL((k_small_down<T, decltype(k4)::value, false, true>), grid, dim3(64), 0, st, A, l);
    });
  with_class(cls, [&](auto k4, auto ex) {
    hipLaunchKernelGGL((k_small_down<T, decltype(k4)::value, decltype(ex)::value, false>), grid, dim3(64), 0, st, A, l);
  });
}
template <typename T>
void launch_forward(int cls, dim3 grid, const SmallArgs<T>& A, int l, bool upd, bool app, hipStream_t st) {
  if (far_rhs<T>(A.n, A.m))
    return with_class(cls & ~1, [&](auto k4, auto) {
      hipLaunchKernelGGL((k_small_forward<T, decltype(k4)::value, false, true>), grid, dim3(64), 0, st, A, l, (int)upd,
                         (int)app);
    });
  with_class(cls, [&](auto k4, auto ex) {
    hipLaunchKernelGGL((k_small_forward<T, decltype(k4)::value, decltype(ex)::value, false>), grid, dim3(64), 0, st, A,
                       l, (int)upd, (int)app);
  });
}
template <typename T>
void launch_tail(int cls, dim3 grid, const SmallArgs<T>& A, int lo, hipStream_t st) {
  with_class(cls, [&](auto k4, auto ex) {
    constexpr int K4 = decltype(k4)::value;
    constexpr bool EX = decltype(ex)::value;
    if constexpr (K4 <= 4) {
      const size_t lds = sizeof(T) * kTailWaves * SmallShape<T, K4, EX>::elems(A.m);
      hipLaunchKernelGGL((k_small_tail<T, K4, EX>), grid, dim3(64 * kTailWaves), lds, st, A, lo);
    }
  });
}

}  // namespace

hipError_t init_small_kernels() {
  hipError_t e = set_small_attrs<float>();
  return e == hipSuccess ? set_small_attrs<double>() : e;
}

int small_class(int n, int m) {
  // one wavefront holds 16 right-hand sides as payload rows, two hold 32
  const int k4 = m > 16 ? std::max(5, (n + 3) / 4) : (n + 3) / 4;
  return 2 * (k4 - 1) + (n == 4 * k4 ? 1 : 0);
}

int small_up_tasks(int N, int n, int m, int l) {
  const Level lv = level_info(N, l);
  const int per = small_class(n, m) < 2 * 4 ? 1 : 2;  // targets per task
  return lv.dim + (l > 0 ? (N / (2 * lv.s) + per - 1) / per : 0);
}

template <typename T>
hipError_t small_up_level(T* L, T* E, T* x, const uint8_t* mask, int B, int N, int n, int m, int l, hipStream_t st,
                          const T* Lsrc, const T* Esrc) {
  if (n > kSmallN) return wide_up_level<T>(L, E, x, mask, B, N, n, m, l, st, Lsrc, Esrc);
  if (B <= 0) return hipSuccess;
  kt_begin(kKcPotrf, st);
  launch_up<T>(small_class(n, x != nullptr ? m : 0), dim3(small_up_tasks(N, n, x != nullptr ? m : 0, l), B),
               regular_args(L, E, x, mask, N, n, m, Lsrc, Esrc), l, st);
  kt_end(kKcPotrf, st);
  return hipGetLastError();
}

// The narrowest levels of systems with one wavefront per task run in
// k_small_tail, up and down, as long as the systems are at most one workgroup
// per compute unit; from the first level of at most 16 tasks.  Measured (FP64
// factor_and_solve, every level a launch / with k_small_tail): n=12 N=20 41.8 /
// 35.5 us, n=12 N=100 57.7 / 52.1, n=10 N=1000 87.6 / 82.9, 256 systems of n=12
// N=40 80.5 / 66.9; 2000 systems of n=4 N=30 117.8 / 154.4.  With two
// wavefronts per task (n > 16) a compute unit holds too few tasks: n=32 N=100
// 102 / 117.  (At n = 13 .. 15 the 1024 threads leave the compiler 9 (FP32) or 12
// (FP64) registers short, which it spills.  Timed in six shapes each, 1 to 256
// systems: n = 12 0.81 to 0.92 of the time by level launches, n = 13 .. 15 0.87 to 0.97,
// n = 16 0.83 to 0.98.)
bool small_tail_applies(int B, int n, int m) {
  return n <= kSmallN && small_class(n, m) < 2 * 4 && B <= kTailMaxSystems;
}

template <typename T>
hipError_t small_factor(T* L, T* E, T* x, const uint8_t* mask, int B, int N, int n, int m, bool back, hipStream_t st,
                        const T* Lsrc, const T* Esrc) {
  if (B <= 0) return hipSuccess;
  const int Lv = recursive_iterations(N);
  if (n > kSmallN) {
    hipError_t e = hipSuccess;
    for (int l = 0; l < Lv && e == hipSuccess; ++l)
      e = wide_up_level<T>(L, E, x, mask, B, N, n, m, l, st, Lsrc, Esrc);
    return e;
  }
  const int mx = x != nullptr ? m : 0, cls = small_class(n, mx);
  const SmallArgs<T> A = regular_args(L, E, x, mask, N, n, m, Lsrc, Esrc);
  int lo = Lv;
  if (small_tail_applies(B, n, mx) && (x == nullptr || back)) {
    lo = 0;
    while (lo < Lv && small_up_tasks(N, n, mx, lo) > kTailWaves) ++lo;
  }
  kt_begin(kKcPotrf, st);
  for (int l = 0; l < lo; ++l) launch_up<T>(cls, dim3(small_up_tasks(N, n, mx, l), B), A, l, st);
  if (lo < Lv) launch_tail<T>(cls, dim3(1, B), A, lo, st);
  kt_end(kKcPotrf, st);
  hipError_t e = hipGetLastError();
  if (x != nullptr && back && small_tail_applies(B, n, mx))
    for (int l = lo - 1; l >= 0 && e == hipSuccess; --l) e = small_backward_level<T>(L, E, x, mask, B, N, n, m, l, st);
  return e;
}

template <typename T>
hipError_t small_forward_step(const T* L, const T* E, T* x, const uint8_t* mask, int B, int N, int n, int m, int step,
                              hipStream_t st, bool update, bool apply) {
  if (B <= 0 || m <= 0) return hipSuccess;
  const int l = step + 1;
  const Level lv = level_info(N, l);
  update = update && l > 0;
  const int tasks = (update || apply ? lv.dim : 0) + (update ? N / (2 * lv.s) : 0);
  if (tasks <= 0) return hipSuccess;
  kt_begin(kKcForward, st);
  launch_forward<T>(small_class(n, 0), dim3(tasks, B, (m + 15) / 16),
                    regular_args(const_cast<T*>(L), const_cast<T*>(E), x, mask, N, n, m, (const T*)nullptr,
                                 (const T*)nullptr),
                    l, update, apply, st);
  kt_end(kKcForward, st);
  return hipGetLastError();
}

template <typename T>
hipError_t small_backward_level(const T* L, const T* E, T* x, const uint8_t* mask, int B, int N, int n, int m,
                                int lidx, hipStream_t st) {
  const Level lv = level_info(N, lidx);
  if (lv.dim <= 0 || B <= 0 || m <= 0) return hipSuccess;
  kt_begin(kKcBackward, st);
  launch_down<T>(small_class(n, 0), dim3(lv.dim, B, (m + 15) / 16),
                 regular_args(const_cast<T*>(L), const_cast<T*>(E), x, mask, N, n, m, (const T*)nullptr,
                              (const T*)nullptr),
                 lidx, st);
  kt_end(kKcBackward, st);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Uneven systems: the same kernels, a launch per level and group of systems
// with one ceil(n / 4), over a list of (system, task) pairs.  (One workgroup
// per system walking its levels leaves the chip idle behind the long systems
// and runs the wide levels of each a few tasks at a time.  FP64
// factor_and_solve of systems of N = 10..200, n = 8..32, the inputs copied in
// first, one workgroup per system / level launches: 4096 systems 11.7 / 6.0 ms,
// 32 systems without a graph 1.92 / 0.32 ms; 512 systems in FP32 2.26 / 0.47 ms.
// Where the horizons are short it is the other way round: choose_batch in
// capi.hip.)
// ---------------------------------------------------------------------------
struct SmallBatch {
  struct Level {
    size_t first = 0, count = 0;  // nodes, then targets (factor: several per task)
    size_t nodes = 0;
  };
  struct Group {
    int cls = 0, mmax = 0, stream = 0;
    std::vector<Level> levels;
  };
  std::vector<Group> groups;  // by decreasing cost
  int2* tasks = nullptr;      // device
};

void small_batch_free(SmallBatch* b) {
  if (b == nullptr) return;
  if (b->tasks) (void)hipFree(b->tasks);
  delete b;
}

static hipError_t fill_batch(SmallBatch* h, const BatchProblem* probs, int count, int op, int streams) {
  const bool fac = op == SOCU_OP_FACTOR || op == SOCU_OP_FACTOR_AND_SOLVE;
  const bool solve = op != SOCU_OP_FACTOR;
  std::vector<int> of[kSmallN / 4];
  double cost[kSmallN / 4] = {};
  for (int k = 0; k < count; ++k) {
    const BatchProblem& P = probs[k];
    const int k4 = small_class(P.n, fac && solve ? P.m : 0) / 2;
    of[k4].push_back(k);
    cost[k4] += (double)P.N * P.n * P.n;
  }
  std::vector<int> by;
  for (int k4 = 0; k4 < kSmallN / 4; ++k4)
    if (!of[k4].empty()) by.push_back(k4);
  std::stable_sort(by.begin(), by.end(), [&](int x, int y) { return cost[x] > cost[y]; });
  std::vector<double> load(streams, 0.0);
  std::vector<int2> tasks;
  for (int k4 : by) {
    SmallBatch::Group G;
    std::vector<int>& sys = of[k4];
    std::stable_sort(sys.begin(), sys.end(), [&](int x, int y) { return probs[x].N > probs[y].N; });
    bool exact = true;
    for (int k : sys) {
      exact = exact && probs[k].n == 4 * (k4 + 1);
      if (solve) G.mmax = std::max(G.mmax, probs[k].m);
    }
    G.cls = 2 * k4 + (exact ? 1 : 0);
    G.stream = (int)(std::min_element(load.begin(), load.end()) - load.begin());
    load[G.stream] += cost[k4];
    const int per = fac && G.cls >= 2 * 4 ? 2 : 1;  // targets per task
    const int Lv = recursive_iterations(probs[sys[0]].N);
    for (int l = 0; l < Lv; ++l) {
      SmallBatch::Level V;
      const int s = 1 << l;
      V.first = tasks.size();
      for (int k : sys)
        for (int t = 0, dim = (probs[k].N + s) / (2 * s); t < dim; ++t) tasks.push_back({k, t});
      V.nodes = tasks.size() - V.first;
      if (l > 0)
        for (int k : sys) {
          const int dim = (probs[k].N + s) / (2 * s);
          for (int u = 0; u * per < probs[k].N / (2 * s); ++u) tasks.push_back({k, dim + u});
        }
      V.count = tasks.size() - V.first;
      G.levels.push_back(V);
    }
    h->groups.push_back(std::move(G));
  }
  hipError_t e = hipMalloc(&h->tasks, std::max<size_t>(1, tasks.size()) * sizeof(int2));
  if (e == hipSuccess) e = hipMemcpy(h->tasks, tasks.data(), tasks.size() * sizeof(int2), hipMemcpyHostToDevice);
  return e;
}

hipError_t small_batch_create(SmallBatch** out, const BatchProblem* probs, int count, int op, int streams) {
  *out = nullptr;
  SmallBatch* h = nullptr;
  hipError_t e = hipErrorOutOfMemory;
  try {  // (the task list takes host memory of its own: about 12 bytes per block row)
    h = new SmallBatch();
    e = fill_batch(h, probs, count, op, streams);
  } catch (const std::bad_alloc&) {
  } catch (const std::length_error&) {
  }
  if (e != hipSuccess) {
    small_batch_free(h);
    return e;
  }
  *out = h;
  return hipSuccess;
}

bool small_batch_uses(const SmallBatch* h, int stream) {
  for (const auto& G : h->groups)
    if (G.stream == stream) return true;
  return false;
}

template <typename T>
static hipError_t batch_enqueue(const SmallBatch* h, const BatchProblem* probs, const uint8_t* mask, int op, int stream,
                                hipStream_t st) {
  const bool fac = op == SOCU_OP_FACTOR || op == SOCU_OP_FACTOR_AND_SOLVE;
  for (const auto& G : h->groups) {
    if (G.stream != stream) continue;
    SmallArgs<T> A = {};
    A.probs = probs;
    A.mask = mask;
    A.solve = op != SOCU_OP_FACTOR;
    A.m = G.mmax;
    // (several launches for a level of more tasks than one takes)
    auto pieces = [&](size_t first, size_t count, auto launch) {
      for (size_t t = 0; t < count; t += kMaxGridTasks) {
        A.tasks = h->tasks + first + t;
        launch(dim3((unsigned)std::min<size_t>(count - t, kMaxGridTasks)));
      }
    };
    for (size_t l = 0; l < G.levels.size(); ++l) {
      const SmallBatch::Level& V = G.levels[l];
      if (fac) pieces(V.first, V.count, [&](dim3 grid) { launch_up<T>(G.cls, grid, A, (int)l, st); });
      else if (op != SOCU_OP_BACKWARD)
        pieces(V.first, V.count, [&](dim3 grid) { launch_forward<T>(G.cls, grid, A, (int)l, true, true, st); });
    }
    if (op != SOCU_OP_FACTOR && op != SOCU_OP_FORWARD)
      for (int l = (int)G.levels.size() - 1; l >= 0; --l)
        pieces(G.levels[l].first, G.levels[l].nodes, [&](dim3 grid) { launch_down<T>(G.cls, grid, A, l, st); });
  }
  return hipGetLastError();
}

hipError_t small_batch_enqueue(const SmallBatch* h, const BatchProblem* dprobs, const uint8_t* mask, int op, int dtype,
                               int stream, hipStream_t st) {
  return dtype == SOCU_DTYPE_F64 ? batch_enqueue<double>(h, dprobs, mask, op, stream, st)
                                 : batch_enqueue<float>(h, dprobs, mask, op, stream, st);
}

template hipError_t small_up_level<float>(float*, float*, float*, const uint8_t*, int, int, int, int, int, hipStream_t,
                                          const float*, const float*);
template hipError_t small_up_level<double>(double*, double*, double*, const uint8_t*, int, int, int, int, int,
                                           hipStream_t, const double*, const double*);
template hipError_t small_factor<float>(float*, float*, float*, const uint8_t*, int, int, int, int, bool, hipStream_t,
                                        const float*, const float*);
template hipError_t small_forward_step<float>(const float*, const float*, float*, const uint8_t*, int, int, int, int, int,
                                            hipStream_t, bool, bool);
template hipError_t small_backward_level<float>(const float*, const float*, float*, const uint8_t*, int, int, int, int, int,
                                              hipStream_t);
template hipError_t small_factor<double>(double*, double*, double*, const uint8_t*, int, int, int, int, bool, hipStream_t,
                                         const double*, const double*);
template hipError_t small_forward_step<double>(const double*, const double*, double*, const uint8_t*, int, int, int, int, int,
                                            hipStream_t, bool, bool);
template hipError_t small_backward_level<double>(const double*, const double*, double*, const uint8_t*, int, int, int, int, int,
                                              hipStream_t);

}  // namespace socu
