// Level-by-level solve sweeps for blocks of 32 < n <= 128, with the explicit
// inverses of the diagonal blocks (U: the transposed inverse in the strict
// upper triangle of L).
//
// Forward step l (levels ascending): for every receiving block j = 2s(u+1)-1
//   y_j -= R_{j-s} y_{j-s} + Lc_{j+s}^T y_{j+s},
//   then, for the nodes j of level l+1 among them:  y_j <- Linv_j y_j
//   (the reference's forward substitution, block_tridiag_solver.py:425-485);
//   the applies of level 0, which no update precedes, are a launch of their own.
// Backward level l (levels descending): for every node i = s-1+2s*t
//   x_i <- Linv_i^T (x_i - R_i^T x_{i+s} - Lc_i x_{i-s})
//   (block_tridiag_solver.py:581-643).
#include "../../include/socu_hip.h"
#include "nd_common.h"
#include "nd_internal.h"
#include "nd_small.h"
#include "nd_tile.h"

namespace socu {

namespace {

// What a launch does: a whole step, the updates alone, or the applies of the
// nodes of level s alone.
enum StepMode { kStepFull = 0, kStepUpdate = 1, kStepApply = 2 };

// One workgroup per (block, 16 right-hand sides), one wavefront per 16-row tile
// of the block (RT of them).  The vectors x_{i+s}, x_{i-s} and t go through LDS;
// each element of a block is used once, by one wavefront, and goes from memory
// to its registers in the MFMA operand layout, every load issued before the
// first product.  Step q covers k = 8 q .. 8 q + 7 by two MFMAs, lane group g
// taking k = 8 q + 2 g + e in MFMA e: rows are then read 64 (FP64) contiguous
// bytes at a time by four lanes with one load each, and every cache line by two
// consecutive loads.
//
// What bounds it: a compute unit's misses.  A launch of one node takes 5.2 us with
// U alone and 3.5 us more per coupling block (n = 100, FP64: 80 KB, 23 bytes/ns;
// their MFMAs take 1.5 us), and no more with 100 nodes, one per compute unit.
// Four wavefronts taking the tiles in turn, with a branch per load, took 42 us a
// forward step and 20 us a backward level there.  FP64 solve n=100 N=200 m=8
// 518 -> 232 us, factor_and_solve n=64 N=1024 m=16 472 -> 442 us, n=128 N=512
// 975 -> 959 us, FP32 n=36 N=100 B=8 197 -> 171 us.
// FAR: 64-bit offsets, for block rows of right-hand sides above 4 GiB.  A variant of
// its own, so that the common one has no instruction for it; that they would cost
// time there was not shown (factor_and_solve n=64 N=1024 m=16: without FAR 441.8 us,
// 64-bit offsets for all 443.2, this variant, whose instructions are those of the
// first, 443.3).
template <typename T, int RT, bool FWD, bool FAR>
__global__ __launch_bounds__(64 * RT) void k_step(const T* __restrict__ L, const T* __restrict__ E,
                                                  T* __restrict__ x, const uint8_t* __restrict__ mask, int N, int n,
                                                  int m, int nE, int s, int off, int mode) {
  constexpr int NP = 16 * RT, Q = 2 * RT, QT = Q - 2;  // QT: the first step of the last tile
  const int b = blockIdx.z;
  if (masked_out(mask, b)) return;
  const int c0 = blockIdx.y * kRhsChunk;
  const int nn = n * n;
  const size_t nm = (size_t)n * m;
  const T* const Eb = E + (size_t)b * nE * nn;
  T* const xb = x + (size_t)b * N * nm + c0;
  const int u = blockIdx.x;
  const bool targets = FWD && mode != kStepApply;
  const int i = targets ? 2 * s * (u + 1) - 1 : s - 1 + 2 * s * u;
  const bool hasT = mode != kStepApply && i + s < N;              // Lc_{i+s} or R_i, used transposed
  const bool hasS = mode != kStepApply && (targets || i >= s);    // R_{i-s} or Lc_i
  const bool inv = FWD ? mode == kStepApply || (mode == kStepFull && (u & 1) == 0) : true;
  const T* const U = L + ((size_t)b * N + i) * nn;
  const T* const MT = Eb + (size_t)(off + i / s) * nn;
  const T* const MS = Eb + (size_t)(off + (i - s) / s) * nn;
  T* const xi = xb + (size_t)i * nm;

  __shared__ T Xp[NP * 16], Xm[NP * 16], Tt[NP * 16];
  const int lane = lane_id(), li = lane & 15, g = lane >> 4, w = wave_uniform();
  // (the triangular products of tiles t and RT - 1 - t add up to the same)
  const int t = w < 4 ? w : RT + 3 - w;
  const int ii = 16 * t + li, ic = min(ii, n - 1);
  const int cl = min(li, m - c0 - 1);
  const int k0 = threadIdx.x >> 4;  // staging: column li, rows k0 + 4 RT p

  T sp[4], sm[4], xd[4], a1[Q][2], a2[Q][2], a3[Q][2];
  if (hasT) {
#pragma unroll
    for (int p = 0; p < 4; ++p) sp[p] = ld_rhs<FAR>(xi + s * nm, min(k0 + 4 * RT * p, n - 1), m, cl);
  }
  if (hasS) {
#pragma unroll
    for (int p = 0; p < 4; ++p) sm[p] = ld_rhs<FAR>(xi - s * nm, min(k0 + 4 * RT * p, n - 1), m, cl);
  }
  auto rows = [&](T(&v)[2], const T* M, int q) {  // v[e] = M[ii][8 q + 2 g + e]
    const int o = ic * n + 8 * q + 2 * g, oc = q < QT ? o : min(o, nn - 2);
    const auto d = ldg2(M, oc);
    v[0] = (q >= QT && o > oc) ? d.y : d.x;
    v[1] = d.y;
  };
  auto cols = [&](T(&v)[2], const T* M, int q) {  // v[e] = M[8 q + 2 g + e][ii]
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int k = 8 * q + 2 * g + e;
      v[e] = ldg(M, (q < QT ? k : min(k, n - 1)) * n + ic);
    }
  };
  if (hasT) {
#pragma unroll
    for (int q = 0; q < Q; ++q) cols(a1[q], MT, q);
  }
  if (hasS) {
#pragma unroll
    for (int q = 0; q < Q; ++q) rows(a2[q], MS, q);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) xd[e] = ld_rhs<FAR>(xi, min(16 * t + Mfma<T>::row(lane, e), n - 1), m, cl);
  T diag = T(1);
  if (inv) {
    diag = ldg(U, ic * (n + 1));
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      if (FWD ? q / 2 <= t : q / 2 >= t) {
        if (FWD) cols(a3[q], U, q);
        else rows(a3[q], U, q);
      }
    }
  }
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int k = k0 + 4 * RT * p;
    if (hasT) Xp[k * 16 + li] = k < n ? sp[p] : T(0);
    if (hasS) Xm[k * 16 + li] = k < n ? sm[p] : T(0);
  }
  __syncthreads();
  // t = x_i - MT^T x_{i+s} - MS x_{i-s}
  typename Mfma<T>::acc_t acc = acc_zero<T>(), acc2 = acc_zero<T>();
  if (hasT) {
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int k = 8 * q + 2 * g + e;
        acc = Mfma<T>::mma((q < QT || k < n) ? a1[q][e] : T(0), Xp[k * 16 + li], acc);
      }
  }
  if (hasS) {
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int k = 8 * q + 2 * g + e;
        acc2 = Mfma<T>::mma((q < QT || k < n) ? a2[q][e] : T(0), Xm[k * 16 + li], acc2);
      }
  }
  mfma_settle<T>();
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int row = 16 * t + Mfma<T>::row(lane, e);
    const T v = row < n ? xd[e] - (acc[e] + acc2[e]) : T(0);
    if (inv) Tt[row * 16 + li] = v;
    else if (row < n && li < m - c0) st_rhs<FAR>(xi, row, m, li, v);
  }
  if (!inv) return;
  __syncthreads();
  // backward: x_i = A t, A(r, k) = U[r][k] (k > r), 1 / L[r][r] (k = r);
  // forward: y_i = A t, A(r, k) = U[k][r] (k < r), 1 / L[r][r] (k = r)
  const T rd = T(1) / diag;
  acc = acc_zero<T>();
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    if (FWD ? q / 2 <= t : q / 2 >= t) {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int k = 8 * q + 2 * g + e;
        T a = (FWD ? k < ii : k > ii && (q < QT || k < n)) ? a3[q][e] : T(0);
        a = k == ii ? rd : a;
        acc = Mfma<T>::mma(a, Tt[k * 16 + li], acc);
      }
    }
  }
  mfma_settle<T>();
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int row = 16 * t + Mfma<T>::row(lane, e);
    if (row < n && li < m - c0) st_rhs<FAR>(xi, row, m, li, acc[e]);
  }
}

template <typename T, bool FWD>
hipError_t launch_step(const T* L, const T* E, T* x, const uint8_t* mask, int B, int N, int n, int m, int blocks,
                       int s, int off, int mode, hipStream_t st) {
  if (n <= kSmallN || n > kMaxN) return hipErrorInvalidValue;
  const int mch = (m + kRhsChunk - 1) / kRhsChunk;
  if (B <= 0 || mch <= 0 || blocks <= 0) return hipSuccess;
  const int nE = (int)off_diag_storage_len(N);
  auto go = [&](auto rt) {
    constexpr int RT = decltype(rt)::value;
    auto k = far_rhs<T>(n, m) ? k_step<T, RT, FWD, true> : k_step<T, RT, FWD, false>;
    hipLaunchKernelGGL(k, dim3(blocks, mch, B), dim3(64 * RT), 0, st, L, E, x, mask, N, n, m, nE, s, off, mode);
  };
  switch ((n + 15) / 16) {
    case 3: go(std::integral_constant<int, 3>{}); break;
    case 4: go(std::integral_constant<int, 4>{}); break;
    case 5: go(std::integral_constant<int, 5>{}); break;
    case 6: go(std::integral_constant<int, 6>{}); break;
    case 7: go(std::integral_constant<int, 7>{}); break;
    default: go(std::integral_constant<int, 8>{}); break;
  }
  return hipGetLastError();
}

}  // namespace

// Step `step`'s updates (`update`) and level step + 1's applies (`apply`), in one
// launch if both.
template <typename T>
hipError_t wide_forward_step(const T* L, const T* E, T* x, const uint8_t* mask, int B, int N, int n, int m, int step,
                             hipStream_t st, bool update, bool apply) {
  kt_begin(kKcForward, st);
  hipError_t e = hipSuccess;
  const Level nx = level_info(N, step + 1);
  if (update && step >= 0) {
    const Level lv = level_info(N, step);
    e = launch_step<T, true>(L, E, x, mask, B, N, n, m, N / (2 * lv.s), lv.s, lv.off,
                             (apply && nx.dim > 0) ? kStepFull : kStepUpdate, st);
  } else if (apply && nx.dim > 0) {
    e = launch_step<T, true>(L, E, x, mask, B, N, n, m, nx.dim, nx.s, nx.off, kStepApply, st);
  }
  kt_end(kKcForward, st);
  return e;
}

template <typename T>
hipError_t wide_backward_level(const T* L, const T* E, T* x, const uint8_t* mask, int B, int N, int n, int m, int lidx,
                               hipStream_t st) {
  const Level lv = level_info(N, lidx);
  kt_begin(kKcBackward, st);
  const hipError_t e = launch_step<T, false>(L, E, x, mask, B, N, n, m, lv.dim, lv.s, lv.off, kStepFull, st);
  kt_end(kKcBackward, st);
  return e;
}

template hipError_t wide_forward_step<float>(const float*, const float*, float*, const uint8_t*, int, int, int, int,
                                             int, hipStream_t, bool, bool);
template hipError_t wide_forward_step<double>(const double*, const double*, double*, const uint8_t*, int, int, int,
                                              int, int, hipStream_t, bool, bool);
template hipError_t wide_backward_level<float>(const float*, const float*, float*, const uint8_t*, int, int, int, int,
                                               int, hipStream_t);
template hipError_t wide_backward_level<double>(const double*, const double*, double*, const uint8_t*, int, int, int,
                                                int, int, hipStream_t);

}  // namespace socu
