// Block sizes kMaxN < n <= kMaxNLarge: the per-node kernels of the ND factor and
// sweeps, on blocks split in two,
//
//   [ A11  .  ]   n1 = 16 ceil(n / 32) rows, n2 = n - n1 <= n1 <= 128,
//   [ A21 A22 ]
//
// so that the halves of the diagonal go through k_potrf_blk (nd_potrf.hip) and
// everything else is products spread over many workgroups (the reference's
// potrf_blocked, socu/blas/potrf.py:97-119, and trsm_rltn / trsm_llnn,
// trsm.py:94-120, 202-228).  With U = L^-T as in the smaller blocks, in the same
// storage, a factor level is
//
//   potrf        L11, U11 <- A11
//   kPanelFirst  L21 = A21 U11;  R1 <- R1 U11;  Lc1 <- U11^T Lc1
//   kPanelUpdate A22 -= L21 L21^T;  R2 -= R1 L21^T;  Lc2 -= L21 Lc1;
//                U12 = -U11 L21^T
//   potrf        L22, U22 <- A22
//   kPanelSecond U12 <- U12 U22;  R2 <- R2 U22;  Lc2 <- U22^T Lc2
//
// (R1, R2: columns of R; Lc1, Lc2: rows of Lc), then the Schur updates
// (k_schur_tile).  For n <= 128, where the diagonal block is factored whole,
// kPanelFirst is the level's products with U (R <- R U, Lc <- U^T Lc).
//
// Measured (FP64, n = 200, levels of few nodes): one workgroup factoring a whole
// block, 32x32 tiles through HBM, took 205 us per level and the products with U 34;
// the five launches take 22 + 7 + 8 + 19 + 7 us.  A sweep's apply took 27 us and its
// update 36 (32-wide chunks, tiles through LDS one by one): 13 and 9.  For n = 128 the
// products with U took 12 us (U staged in LDS by each of 8 workgroups per node): 7.
// What bounds them now: the halves' pivot chains (see nd_potrf.hip); the products'
// launches, their loads (one compute unit's misses, 23 bytes/ns).  FP64 factor_and_solve
// n=200 N=64 m=2: 2468 -> 1062 us (868 with the Schur tiles).
#include <algorithm>

#include "../../include/socu_hip.h"
#include "nd_common.h"
#include "nd_internal.h"
#include "nd_small.h"
#include "nd_tile.h"

namespace socu {

namespace {

constexpr int kPP = 17;  // pitch of a staged chunk: 16 columns

int first_half(int n) { return n > kMaxN ? 16 * ((n + 31) / 32) : n; }

// The left operand of a product, A(r, k), from a row-major matrix M.
enum LeftForm {
  kRows,     // M[r][k]
  kCols,     // M[k][r]
  kTriRows,  // U = L^-T of a factored block M: M[r][k] for k > r, 1 / M[r][r]
  kTriCols   // U^T: M[k][r] for k < r, 1 / M[r][r]
};

// acc += A(r0 + i, k) X(k, c) over k0 <= k < k1 (k0 a multiple of 32; A zero outside
// its R x K).  X: 16 columns in LDS.  TR: the transposed product, D(c, i).
// Batches of 32 k, the next one's loads issued before the current one's MFMAs;
// lane group g takes k = 8 q + 2 g + e in MFMA (q, e), so that rows are read 64
// bytes (FP64) at a time by four lanes with one load each.
template <typename T, int FORM, bool TR>
__device__ __forceinline__ void panel_mma(typename Mfma<T>::acc_t& acc, const T* M, int ld, int R, int K, int r0,
                                          const T* X, int k0, int k1) {
  const int lane = lane_id(), li = lane & 15, g = lane >> 4;
  const int r = r0 + li, rc = min(r, R - 1);
  constexpr bool tri = FORM == kTriRows || FORM == kTriCols, rows = FORM == kRows || FORM == kTriRows;
  T rd = T(0);
  if constexpr (tri) rd = T(1) / ldg(M, rc * (ld + 1));
  T cur[4][2], nxt[4][2];
  auto load = [&](T(&v)[4][2], int kb) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int k = kb + 8 * q + 2 * g;
      if constexpr (rows) {
        const int kc = min(k, K - 2);
        const auto d = ldg2(M, rc * ld + kc);
        v[q][0] = k > kc ? d.y : d.x;
        v[q][1] = d.y;
      } else {
        v[q][0] = ldg(M, min(k, K - 1) * ld + rc);
        v[q][1] = ldg(M, min(k + 1, K - 1) * ld + rc);
      }
    }
  };
  load(cur, k0);
  for (int kb = k0; kb < k1; kb += 32) {
    if (kb + 32 < k1) load(nxt, kb + 32);
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int k = kb + 8 * q + 2 * g + e;
        bool in = k < K;
        if (FORM == kTriRows) in = in && k > r;
        if (FORM == kTriCols) in = k < r;
        T a = in ? cur[q][e] : T(0);
        if constexpr (tri) a = k == r ? rd : a;
        const T x = X[k * kPP + li];
        acc = TR ? Mfma<T>::mma(x, a, acc) : Mfma<T>::mma(a, x, acc);
      }
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int e = 0; e < 2; ++e) cur[q][e] = nxt[q][e];
  }
  mfma_settle<T>();
}

// A chunk of up to 16 vectors of length K: element k of vector c is p[c * ld + k]
// (rows) or p[k * ld + c].
template <typename T>
struct Chunk {
  T* p;
  int ld, count;
  bool rows;
};

// X(k, c) <- the chunk, zero to 16 columns and to a multiple of 32 in k.  FAR (here
// and below): a chunk of right-hand sides of a block row above 4 GiB (64-bit offsets
// for all cost 0.4% of a factor_and_solve of n=200 N=64 m=2).
template <typename T, int THREADS, bool FAR = false>
__device__ __forceinline__ void stage_chunk(T* X, const Chunk<T>& c, int K) {
  const int kp = (K + 31) & ~31;
#pragma unroll 4
  for (int idx = threadIdx.x; idx < 16 * kp; idx += THREADS) {
    int k, j;
    if (c.rows) {  // 32 consecutive k of a row
      k = (idx & 31) + 32 * (idx >> 9);
      j = (idx >> 5) & 15;
    } else {
      k = idx >> 4;
      j = idx & 15;
    }
    const int kc = min(k, K - 1), jc = min(j, c.count - 1);
    const T v = FAR ? ld_rhs<true>(c.p, kc, c.ld, jc) : ldg(c.p, c.rows ? jc * c.ld + kc : kc * c.ld + jc);
    X[k * kPP + j] = (k < K && j < c.count) ? v : T(0);
  }
}

// out(r, c) = A X (mode 0), -A X (1) or out - A X (2), row tiles t0 + wavefront, ...
// of R rows; lower: rows r >= ... of a symmetric result only up to tile tmax.
template <typename T, int FORM, bool TR, int TH, bool FAR = false>
__device__ __forceinline__ void panel_product(const T* M, int ld, int R, int K, const T* X, const Chunk<T>& out,
                                              int mode, int tmax) {
  const int lane = lane_id(), li = lane & 15, w = wave_uniform();
  for (int t = w; t < tmax; t += TH / 64) {
    typename Mfma<T>::acc_t acc = acc_zero<T>();
    int off[4];
    T c[4];
    bool ok[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = TR ? li : Mfma<T>::row(lane, e), j = TR ? Mfma<T>::row(lane, e) : li;
      ok[e] = 16 * t + i < R && j < out.count;
      const int r = min(16 * t + i, R - 1), jc = min(j, out.count - 1);
      off[e] = TR ? jc * out.ld + r : r * out.ld + jc;
      c[e] = T(0);
    }
    if (mode == 2) {
#pragma unroll
      for (int e = 0; e < 4; ++e) c[e] = ldg(out.p, off[e]);
    }
    const int k0 = FORM == kTriRows ? (16 * t) & ~31 : 0, k1 = FORM == kTriCols ? min(16 * t + 16, K) : K;
    panel_mma<T, FORM, TR>(acc, M, ld, R, K, 16 * t, X, k0, k1);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (ok[e]) {
        if constexpr (FAR) st_rhs<true>(out.p, 16 * t + Mfma<T>::row(lane, e), out.ld, li, acc[e]);  // (mode 0, not TR)
        else stg(out.p, off[e], mode == 0 ? acc[e] : c[e] - acc[e]);
      }
  }
}

enum PanelPhase { kPanelFirst, kPanelUpdate, kPanelSecond, kPanelInverse, kPanelInverseSecond, kPanelForward, kPanelBackward };

// Workgroup (node, chunk of 16 vectors): see above.  kPanelInverse and
// kPanelInverseSecond: the U12 products alone, for every block (s = 0), L21 being
// read from Lsrc; kPanelForward / kPanelBackward: x_i <- U^T x_i / U x_i.
template <typename T, int TH, bool FAR>
__global__ __launch_bounds__(TH) void k_large_panel(T* L, const T* Lsrc, T* E, const T* Esrc, T* x,
                                                              const uint8_t* __restrict__ mask, int N, int n, int n1,
                                                              int m, int nE, int s, int off, int phase) {
  __shared__ T X[kMaxNLarge * kPP];
  const int b = blockIdx.z;
  if (masked_out(mask, b)) return;
  const int i = s > 0 ? s - 1 + 2 * s * blockIdx.x : blockIdx.x;
  const size_t nn = (size_t)n * n;
  T* const A = L + ((size_t)b * N + i) * nn;
  T* const Eb = E + (size_t)b * nE * nn;
  const int n2 = n - n1, c1 = (n1 + 15) / 16, c2 = (n2 + 15) / 16, cn = (n + 15) / 16;
  int y = blockIdx.y;

  if (phase == kPanelForward || phase == kPanelBackward) {
    const int c0 = 16 * y;
    const Chunk<T> v{x + ((size_t)b * N + i) * n * m + c0, m, min(16, m - c0), false};
    stage_chunk<T, TH, FAR>(X, v, n);
    __syncthreads();
    if (phase == kPanelForward) panel_product<T, kTriCols, false, TH, FAR>(A, n, n, n, X, v, 0, cn);
    else panel_product<T, kTriRows, false, TH, FAR>(A, n, n, n, X, v, 0, cn);
    return;
  }
  if (phase == kPanelInverse || phase == kPanelUpdate) {
    const T* const L21 = (phase == kPanelInverse ? Lsrc + (A - L) : A) + (size_t)n1 * n;
    // (what a chunk reads and writes does not overlap: the cast is for its type)
    if (y < c2) {  // U12 columns 16 y ..
      const Chunk<T> v{const_cast<T*>(L21) + (size_t)16 * y * n, n, min(16, n2 - 16 * y), true};
      stage_chunk<T, TH>(X, v, n1);
      __syncthreads();
      const Chunk<T> o{A + n1 + 16 * y, n, v.count, false};
      panel_product<T, kTriRows, false, TH>(A, n, n1, n1, X, o, 1, c1);
      return;
    }
    y -= c2;
    if (y < c2) {  // A22 rows 16 y .., up to their diagonal tile
      const Chunk<T> v{const_cast<T*>(L21) + (size_t)16 * y * n, n, min(16, n2 - 16 * y), true};
      stage_chunk<T, TH>(X, v, n1);
      __syncthreads();
      const Chunk<T> o{A + (size_t)(n1 + 16 * y) * n + n1, n, v.count, true};
      panel_product<T, kRows, true, TH>(L21, n, n2, n1, X, o, 2, y + 1);
      return;
    }
    y -= c2;
    if (y < cn) {  // R rows
      if (i + s >= N) return;
      T* const R = Eb + (size_t)(off + i / s) * nn + (size_t)16 * y * n;
      const Chunk<T> v{R, n, min(16, n - 16 * y), true}, o{R + n1, n, v.count, true};
      stage_chunk<T, TH>(X, v, n1);
      __syncthreads();
      panel_product<T, kRows, true, TH>(L21, n, n2, n1, X, o, 2, c2);
      return;
    }
    y -= cn;
    if (i < s) return;
    T* const C = Eb + (size_t)(off + (i - s) / s) * nn + 16 * y;  // Lc columns
    const Chunk<T> v{C, n, min(16, n - 16 * y), false}, o{C + (size_t)n1 * n, n, v.count, false};
    stage_chunk<T, TH>(X, v, n1);
    __syncthreads();
    panel_product<T, kRows, false, TH>(L21, n, n2, n1, X, o, 2, c2);
    return;
  }
  // products with U11 (kPanelFirst) or U22, in place
  const bool first = phase == kPanelFirst;
  const int K = first ? n1 : n2, h = first ? 0 : n1, ct = first ? c2 : c1;
  const T* const U = A + (size_t)h * (n + 1);
  Chunk<T> v;
  if (y < ct) {  // L21 rows / U12 rows
    v = Chunk<T>{(first ? A + (size_t)n1 * n : A + n1) + (size_t)16 * y * n, n, min(16, (first ? n2 : n1) - 16 * y), true};
  } else if (y - ct < cn) {
    if (i + s >= N) return;
    y -= ct;
    v = Chunk<T>{Eb + (size_t)(off + i / s) * nn + (size_t)16 * y * n + h, n, min(16, n - 16 * y), true};
  } else {
    if (i < s) return;
    y -= ct + cn;
    v = Chunk<T>{Eb + (size_t)(off + (i - s) / s) * nn + (size_t)h * n + 16 * y, n, min(16, n - 16 * y), false};
  }
  Chunk<T> in = v;
  if (Esrc != nullptr) in.p = const_cast<T*>(Esrc) + (v.p - E);  // (R and Lc alone: n <= kMaxN)
  stage_chunk<T, TH>(X, in, K);
  __syncthreads();
  if (v.rows) panel_product<T, kTriCols, true, TH>(U, n, K, K, X, v, 0, (K + 15) / 16);
  else panel_product<T, kTriCols, false, TH>(U, n, K, K, X, v, 0, (K + 15) / 16);
}

// Sweep updates, one workgroup per (block, 16-row tile, 16 right-hand sides), grid
// (items, row tiles * chunks, B); wavefronts 0, 1 take the halves of one product's
// K, 2, 3 those of the other.
//   forward (target j = 2s(u+1)-1): y_j -= R_{j-s} y_{j-s} + Lc_{j+s}^T y_{j+s}
//   backward (node i = s-1+2su):    x_i -= Lc_i x_{i-s} + R_i^T x_{i+s}
// (gemm_nn / gemm_tn, gemm.py:151-201, :358-408)
template <typename T, bool BWD, bool FAR>
__global__ __launch_bounds__(kThreads) void k_update_large(const T* __restrict__ E, T* __restrict__ x,
                                                          const uint8_t* __restrict__ mask, int N, int n, int m,
                                                          int nE, int s, int off) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ T part[4][256];
  T* const Xa = reinterpret_cast<T*>(smem_raw);
  T* const Xc = Xa + ((n + 31) & ~31) * kPP;
  const int b = blockIdx.z;
  if (masked_out(mask, b)) return;
  const int tiles = (n + 15) / 16, t = blockIdx.y % tiles, c0 = 16 * (blockIdx.y / tiles);
  const size_t nn = (size_t)n * n, nm = (size_t)n * m;
  const T* const Eb = E + (size_t)b * nE * nn;
  T* const xb = x + (size_t)b * N * nm + c0;
  const int j = BWD ? s - 1 + 2 * s * blockIdx.x : 2 * s * (blockIdx.x + 1) - 1;
  const bool below = BWD ? j >= s : true, above = j + s < N;
  if (!below && !above) return;
  const int lane = lane_id(), w = wave_uniform(), count = min(16, m - c0);
  const T* const Ma = Eb + (size_t)(off + (j - s) / s) * nn;  // block (j, j-s)
  const T* const Mc = Eb + (size_t)(off + j / s) * nn;        // block (j+s, j)
  if (below) stage_chunk<T, kThreads, FAR>(Xa, Chunk<T>{xb + (j - s) * nm, m, count, false}, n);
  if (above) stage_chunk<T, kThreads, FAR>(Xc, Chunk<T>{xb + (j + s) * nm, m, count, false}, n);
  __syncthreads();
  const int half = (n / 2 + 31) & ~31, k0 = (w & 1) ? half : 0, k1 = (w & 1) ? n : half;
  typename Mfma<T>::acc_t acc = acc_zero<T>();
  if (w < 2) {
    if (below) panel_mma<T, kRows, false>(acc, Ma, n, n, k1, 16 * t, Xa, k0, k1);
  } else {
    if (above) panel_mma<T, kCols, false>(acc, Mc, n, n, k1, 16 * t, Xc, k0, k1);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) part[w][e * 64 + lane] = acc[e];
  __syncthreads();
  // entry e = w of the tile's accumulator layout
  const int row = 16 * t + Mfma<T>::row(lane, w), col = lane & 15;
  const int q = w * 64 + lane;
  if (row < n && col < count) {
    T* const p = xb + j * nm;
    const T sum = (part[0][q] + part[1][q]) + (part[2][q] + part[3][q]);
    st_rhs<FAR>(p, row, m, col, ld_rhs<FAR>(p, row, m, col) - sum);
  }
}

// Schur updates, one workgroup per 16x16 output tile, grid
// (tasks, B):
//   targets   j = 2s(u+1)-1, tiles tc <= tr:  L_j -= R R^T + Lc^T Lc
//   fill-ins  of node i = s-1+2s(f+1):        F = -R Lc
// (syrk.py, gemm.py).  The wavefronts share the sum: a half of K of one product
// each, or a quarter of R Lc.  Both operands go from memory to registers in the
// operand layout.  k_schur_blk's 64x64 tiles walk K with a barrier per 32 columns
// and leave most of the chip idle on a level of few nodes: n = 200, FP64, levels of
// 32, 16, 8, 4, 2 nodes 76, 62, 40, 47, 53 -> 54, 29, 17, 10, 7 us (the larger ones
// at 6.7 ns a tile, 19 TFLOP/s).  FP64 factor_and_solve n=200 N=64 m=2 1059 -> 868 us,
// n=128 N=512 896 -> 881 us.
template <typename T, bool COLS>
__device__ __forceinline__ void pair_load(T (&v)[4][2], const T* M, int n, int rc, int kb, int g) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int k = kb + 8 * q + 2 * g;
    if constexpr (COLS) {
      v[q][0] = ldg(M, min(k, n - 1) * n + rc);
      v[q][1] = ldg(M, min(k + 1, n - 1) * n + rc);
    } else {
      const int kc = min(k, n - 2);
      const auto d = ldg2(M, rc * n + kc);
      v[q][0] = k > kc ? d.y : d.x;
      v[q][1] = d.y;
    }
  }
}

template <typename T, bool ACOLS, bool BCOLS>
__device__ __forceinline__ void pair_mma(typename Mfma<T>::acc_t& acc, const T* A, const T* B, int n, int r0, int c0,
                                         int k0, int k1) {
  const int lane = lane_id(), g = lane >> 4;
  const int rc = min(r0 + (lane & 15), n - 1), cc = min(c0 + (lane & 15), n - 1);
  T a[4][2], b[4][2], na[4][2], nb[4][2];
  pair_load<T, ACOLS>(a, A, n, rc, k0, g);
  pair_load<T, BCOLS>(b, B, n, cc, k0, g);
  for (int kb = k0; kb < k1; kb += 32) {
    if (kb + 32 < k1) {
      pair_load<T, ACOLS>(na, A, n, rc, kb + 32, g);
      pair_load<T, BCOLS>(nb, B, n, cc, kb + 32, g);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const bool in = kb + 8 * q + 2 * g + e < k1;
        acc = Mfma<T>::mma(in ? a[q][e] : T(0), in ? b[q][e] : T(0), acc);
        a[q][e] = na[q][e];
        b[q][e] = nb[q][e];
      }
  }
  mfma_settle<T>();
}

// (ONE: n = 1, where a row holds no pair; its transpose is read instead)
template <typename T, bool ONE>
__global__ __launch_bounds__(kThreads) void k_schur_tile(T* L, const T* Lsrc, T* E,
                                                        const uint8_t* __restrict__ mask, int N, int n,
                                                        int nE, int s, int off, int next_off, int nT, int first) {
  __shared__ T part[4][256];
  const int b = blockIdx.y;
  if (masked_out(mask, b)) return;
  const int nt = (n + 15) / 16, ntri = nt * (nt + 1) / 2;
  const size_t nn = (size_t)n * n;
  T* const Eb = E + (size_t)b * nE * nn;
  const int lane = lane_id(), w = wave_uniform();
  int task = first + blockIdx.x, tr, tc;
  T* C;
  const bool target = task < nT * ntri;
  typename Mfma<T>::acc_t acc = acc_zero<T>();
  if (target) {
    const int j = 2 * s * (task / ntri + 1) - 1;
    tc = task % ntri;
    tr = 0;
    while (tc > tr) tc -= ++tr;
    C = L + ((size_t)b * N + j) * nn;
    const T* const R = Eb + (size_t)(off + (j - s) / s) * nn;
    const T* const Lc = Eb + (size_t)(off + j / s) * nn;
    const int half = (n / 2 + 7) & ~7, k0 = (w & 1) ? half : 0, k1 = (w & 1) ? n : min(half, n);
    if (w < 2) pair_mma<T, ONE, ONE>(acc, R, R, n, 16 * tr, 16 * tc, k0, k1);
    else if (j + s < N) pair_mma<T, true, true>(acc, Lc, Lc, n, 16 * tr, 16 * tc, k0, k1);
  } else {
    task -= nT * ntri;
    const int i = s - 1 + 2 * s * (task / (nt * nt) + 1);
    const int q = task % (nt * nt);
    tr = q / nt;
    tc = q % nt;
    C = Eb + (size_t)(next_off + (i - s) / (2 * s)) * nn;
    const int part4 = (n / 4 + 7) & ~7, k0 = w * part4, k1 = w == 3 ? n : min(k0 + part4, n);
    pair_mma<T, ONE, true>(acc, Eb + (size_t)(off + i / s) * nn, Eb + (size_t)(off + (i - s) / s) * nn, n, 16 * tr,
                             16 * tc, k0, k1);
  }
  const int row = 16 * tr + Mfma<T>::row(lane, w), col = 16 * tc + (lane & 15);
  const bool in = row < n && col < n && (!target || col <= row);
  // (the fill-in block's contents on entry are not read: this is its only update)
  const T c = target && in ? ldg(Lsrc != nullptr ? Lsrc + (C - L) : C, row * n + col) : T(0);
#pragma unroll
  for (int e = 0; e < 4; ++e) part[w][e * 64 + lane] = acc[e];
  __syncthreads();
  const int q = w * 64 + lane;
  if (in) stg(C, row * n + col, c - ((part[0][q] + part[1][q]) + (part[2][q] + part[3][q])));
}

template <typename T>
constexpr size_t update_lds(int n) {
  return sizeof(T) * 2 * ((n + 31) & ~31) * kPP;
}

template <typename T>
hipError_t set_attrs() {
  hipError_t e = hipSuccess;
  for (const void* k : {(const void*)k_update_large<T, false, false>, (const void*)k_update_large<T, false, true>,
                        (const void*)k_update_large<T, true, false>, (const void*)k_update_large<T, true, true>})
    if (e == hipSuccess) e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)update_lds<T>(kMaxNLarge));
  return e;
}

template <typename T>
hipError_t launch_panel(T* L, const T* Lsrc, T* E, const T* Esrc, T* x, const uint8_t* mask, int B, int N, int n,
                        int m, int nodes, int chunks, int s, int off, int phase, hipStream_t st) {
  if (nodes <= 0 || chunks <= 0 || B <= 0) return hipSuccess;
  auto go = [&](auto th) {
    constexpr int TH = decltype(th)::value;
    auto k = x != nullptr && far_rhs<T>(n, m) ? k_large_panel<T, TH, true> : k_large_panel<T, TH, false>;
    hipLaunchKernelGGL(k, dim3(nodes, chunks, B), dim3(TH), 0, st, L, Lsrc, E, Esrc, x, mask, N, n, first_half(n), m,
                       (int)off_diag_storage_len(N), s, off, phase);
  };
  // (a wavefront per 16-row tile, up to eight)
  if (n <= 32) go(std::integral_constant<int, 128>{});
  else if (n <= 64) go(std::integral_constant<int, 256>{});
  else go(std::integral_constant<int, 512>{});
  return hipGetLastError();
}

}  // namespace

hipError_t init_large_kernels() {
  const hipError_t e = set_attrs<float>();
  return e == hipSuccess ? set_attrs<double>() : e;
}

// The factor of a level's blocks and, unless it is the last level, its R and Lc.
template <typename T>
hipError_t factor_large(T* L, T* E, const uint8_t* mask, int B, int N, int n, int lidx, hipStream_t st) {
  const Level lv = level_info(N, lidx);
  if (lv.dim <= 0 || B <= 0) return hipSuccess;
  const int n1 = first_half(n), n2 = n - n1, c1 = (n1 + 15) / 16, c2 = (n2 + 15) / 16;
  const int ce = lidx == recursive_iterations(N) - 1 ? 0 : 2 * ((n + 15) / 16);
  T* const none = nullptr;
  hipError_t e = potrf_level<T>(L, mask, B, N, n, lidx, false, none, 0, n1, st);
  kt_begin(kKcTrsm, st);
  if (e == hipSuccess)
    e = launch_panel<T>(L, none, E, none, none, mask, B, N, n, 1, lv.dim, c2 + ce, lv.s, lv.off, kPanelFirst, st);
  if (e == hipSuccess)
    e = launch_panel<T>(L, none, E, none, none, mask, B, N, n, 1, lv.dim, 2 * c2 + ce, lv.s, lv.off, kPanelUpdate, st);
  kt_end(kKcTrsm, st);
  if (e == hipSuccess) e = potrf_level<T>(L, mask, B, N, n, lidx, false, none, n1, n2, st);
  kt_begin(kKcTrsm, st);
  if (e == hipSuccess)
    e = launch_panel<T>(L, none, E, none, none, mask, B, N, n, 1, lv.dim, c1 + ce, lv.s, lv.off, kPanelSecond, st);
  kt_end(kKcTrsm, st);
  return e;
}

template <typename T>
hipError_t schur_tiles(T* L, const T* Lsrc, T* E, const uint8_t* mask, int B, int N, int n, int lidx, int nT, int nF,
                       hipStream_t st) {
  const Level lv = level_info(N, lidx);
  const int nt = (n + 15) / 16, tasks = nT * (nt * (nt + 1) / 2) + nF * nt * nt;
  if (tasks <= 0 || B <= 0) return hipSuccess;
  auto k = n > 1 ? k_schur_tile<T, false> : k_schur_tile<T, true>;
  // (a launch takes 2^32 threads along x; the 32x32 tiles of long systems of small
  // blocks are four times as many 16x16 ones)
  for (int first = 0; first < tasks; first += kMaxGridTasks)
    hipLaunchKernelGGL(k, dim3(std::min(tasks - first, kMaxGridTasks), B), dim3(kThreads), 0, st, L, Lsrc, E, mask, N, n,
                       (int)off_diag_storage_len(N), lv.s, lv.off, lv.next_off, nT, first);
  return hipGetLastError();
}

template <typename T>
hipError_t trsm_level(const T* L, T* E, const T* Esrc, const uint8_t* mask, int B, int N, int n, int lidx,
                      hipStream_t st) {
  if (n > kMaxN) return hipErrorInvalidValue;
  const Level lv = level_info(N, lidx);
  kt_begin(kKcTrsm, st);
  const hipError_t e = launch_panel<T>(const_cast<T*>(L), nullptr, E, Esrc, nullptr, mask, B, N, n, 1, lv.dim,
                                       2 * ((n + 15) / 16), lv.s, lv.off, kPanelFirst, st);
  kt_end(kKcTrsm, st);
  return e;
}

template <typename T>
hipError_t apply_large(const T* L, T* x, const uint8_t* mask, int B, int N, int n, int m, int lidx, bool bwd,
                       hipStream_t st) {
  const Level lv = level_info(N, lidx);
  // (L is only read in these phases)
  return launch_panel<T>(const_cast<T*>(L), nullptr, nullptr, nullptr, x, mask, B, N, n, m, lv.dim, (m + 15) / 16, lv.s, 0,
                         bwd ? kPanelBackward : kPanelForward, st);
}

template <typename T>
hipError_t update_large(const T* E, T* x, const uint8_t* mask, int B, int N, int n, int m, int lidx, bool bwd,
                        hipStream_t st) {
  const Level lv = level_info(N, lidx);
  const int items = bwd ? lv.dim : N / (2 * lv.s);
  if (items <= 0 || B <= 0) return hipSuccess;
  const dim3 grid(items, ((n + 15) / 16) * ((m + 15) / 16), B);
  const int nE = (int)off_diag_storage_len(N);
  auto k = far_rhs<T>(n, m) ? (bwd ? k_update_large<T, true, true> : k_update_large<T, false, true>)
                            : (bwd ? k_update_large<T, true, false> : k_update_large<T, false, false>);
  hipLaunchKernelGGL(k, grid, dim3(kThreads), update_lds<T>(n), st, E, x, mask, N, n, m, nE, lv.s, lv.off);
  return hipGetLastError();
}

// W: U of every block, from tril(L) alone (the rest of W is not written, but for the
// diagonal tiles' triangles).
template <typename T>
hipError_t trtri_large(const T* L, T* W, const uint8_t* mask, int B, int N, int n, hipStream_t st) {
  const int n1 = first_half(n), n2 = n - n1;
  T* const none = nullptr;
  hipError_t e = trtri_blocks<T>(L, W, mask, B, N, n, 0, n1, st);
  if (e == hipSuccess) e = trtri_blocks<T>(L, W, mask, B, N, n, n1, n2, st);
  if (e == hipSuccess)
    e = launch_panel<T>(W, L, none, none, none, mask, B, N, n, 1, N, (n2 + 15) / 16, 0, 0, kPanelInverse, st);
  if (e == hipSuccess)
    e = launch_panel<T>(W, none, none, none, none, mask, B, N, n, 1, N, (n1 + 15) / 16, 0, 0, kPanelInverseSecond, st);
  return e;
}

template hipError_t factor_large<float>(float*, float*, const uint8_t*, int, int, int, int, hipStream_t);
template hipError_t factor_large<double>(double*, double*, const uint8_t*, int, int, int, int, hipStream_t);
template hipError_t schur_tiles<float>(float*, const float*, float*, const uint8_t*, int, int, int, int, int, int,
                                       hipStream_t);
template hipError_t schur_tiles<double>(double*, const double*, double*, const uint8_t*, int, int, int, int, int, int,
                                        hipStream_t);
template hipError_t trsm_level<float>(const float*, float*, const float*, const uint8_t*, int, int, int, int, hipStream_t);
template hipError_t trsm_level<double>(const double*, double*, const double*, const uint8_t*, int, int, int, int,
                                       hipStream_t);
template hipError_t apply_large<float>(const float*, float*, const uint8_t*, int, int, int, int, int, bool,
                                       hipStream_t);
template hipError_t apply_large<double>(const double*, double*, const uint8_t*, int, int, int, int, int, bool,
                                        hipStream_t);
template hipError_t update_large<float>(const float*, float*, const uint8_t*, int, int, int, int, int, bool,
                                        hipStream_t);
template hipError_t update_large<double>(const double*, double*, const uint8_t*, int, int, int, int, int, bool,
                                         hipStream_t);
template hipError_t trtri_large<float>(const float*, float*, const uint8_t*, int, int, int, hipStream_t);
template hipError_t trtri_large<double>(const double*, double*, const uint8_t*, int, int, int, hipStream_t);

}  // namespace socu
