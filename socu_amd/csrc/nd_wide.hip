// Factor levels of blocks of 32 < n <= 64, one launch per level: the node and
// target tasks of nd_small.hip by four wavefronts.
//
// Each wavefront owns one set of payload rows of the panel factor (nd_panel.h)
// and keeps them in registers, as MFMA accumulators, from the updates that
// form them to the panel that finishes them:
//   0  the block's own rows: rows of L_k below the panel's diagonal tile, of
//      U = L_k^-T above it, of the identity at it;
//   1  R_k;   2  Lc_k^T;   3  y_k^T (up to 64 right-hand sides).
// Per panel of 16 columns: its column tile goes through LDS into the
// one-row-per-lane form, the panel runs (every wavefront factors the 16x16
// diagonal tile itself), the result goes through LDS into the operand form,
// and MFMA updates the column tiles to the right in place.
// The operands of the updates from the level below are staged in LDS by
// coalesced loads, shared by the wavefronts.
//
// What bounds it: one task's latency (one workgroup per compute unit at
// n = 64).  FP64, n = 64, a node with both couplings: 62k cycles, of which 6.5k
// the staging, 25k the products (an FP64 MFMA takes 64 cycles; wavefront 0 has
// 320 of them) and 7.5k per panel (pivot chain and LDS 3.3k, MFMA update 3.8k).
// With the payload rows in LDS, updated tile by tile, a panel took 10k, and with
// operands read from global memory in the operand layout (16 cache lines per
// load) the products 46k.  Launches of one node: 27 us at n = 64, 17 at n = 34,
// 13 at n = 36 in FP32, where the separate factor, trsm and Schur launches of a
// level took 31, 26 and 27.  FP64 factor_and_solve n=64 N=1024 m=16 590 -> 472 us,
// n=34 N=128 (two launches) 297 -> 224 us, FP32 n=36 N=100 B=8 eager 340 -> 196 us.
#include "../../include/socu_hip.h"
#include "nd_common.h"
#include "nd_internal.h"
#include "nd_small.h"
#include "nd_tile.h"

namespace socu {

namespace {

constexpr int kWideThreads = 256;

// K4 = n / 4 rounded up to the next even number, EX: n == 4 K4.
template <typename T, int K4, bool EX>
struct WideShape {
  static constexpr int NB = (K4 + 3) / 4;
  static constexpr int NC = 4 * K4 - 16 * (NB - 1);  // columns of the last panel
  static constexpr int NP = 16 * NB;
  static constexpr int SP = NP + 1;      // pitch of a staged block
  static constexpr int kBlock = NP * SP;
  static constexpr int XP = 17;          // pitch of a column tile
  static constexpr int kX = 64 * XP;     // a wavefront's column tile
  // two of wavefront 0's, one each of the others', U_kk, identity
  static constexpr int kFactor = 5 * kX + 16 * XP + 32;
  static constexpr int elems(int blocks) { return blocks * kBlock > kFactor ? blocks * kBlock : kFactor; }
};

// A wavefront's payload rows: [row tile][column tile].
template <typename T, int K4>
using WideAcc = typename Mfma<T>::acc_t[4][(K4 + 3) / 4];

// A block into LDS by the whole workgroup, zero padded: loads, then stores.
template <typename T, int K4, bool EX>
struct Staged {
  using Sh = WideShape<T, K4, EX>;
  T v[Sh::NP / 4];
  __device__ __forceinline__ void load(const T* M, int n, int w) {
    const int c = min(lane_id(), n - 1);
#pragma unroll
    for (int e = 0; e < Sh::NP / 4; ++e) v[e] = ldg(M, min(w + 4 * e, n - 1) * n + c);
  }
  __device__ __forceinline__ void store(T* B, int n, int w) {
    const int c = lane_id();
    if (Sh::NP < 64 && c >= Sh::NP) return;
#pragma unroll
    for (int e = 0; e < Sh::NP / 4; ++e) {
      const int r = w + 4 * e;
      T x = v[e];
      if (!EX || 4 * K4 < Sh::NP) x = (r < n && c < n) ? x : T(0);
      B[r * Sh::SP + c] = x;
    }
  }
};

// acc(i, j) -= sum_k A(i, k) B(k, j) over the block's tiles, operands from two
// staged blocks: A(i, k) = Ab[i][k], or Ab[k][i] (AT); B(k, j) = Bb[j][k] (BT), or
// Bb[k][j].  LOWER: the tiles j <= i only.
template <typename T, int K4, bool EX, bool AT, bool BT, bool LOWER>
__device__ __forceinline__ void staged_mma(WideAcc<T, K4>& acc, const T* Ab, const T* Bb) {
  using Sh = WideShape<T, K4, EX>;
  constexpr int NB = Sh::NB, SP = Sh::SP;
  const int r = lane_id() & 15, g = lane_id() >> 4;
  const T* a0 = Ab + (AT ? g * SP + r : r * SP + g);
  const T* b0 = Bb + (BT ? r * SP + g : g * SP + r);
  // (unrolled: in a loop the compiler carries the accumulators in vector
  // registers and copies them to accumulation registers and back per step)
#pragma unroll
  for (int t = 0; t < K4; ++t) {
    T a[NB], b[NB];
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      a[q] = -a0[AT ? 4 * t * SP + 16 * q : 16 * q * SP + 4 * t];
      b[q] = b0[BT ? 16 * q * SP + 4 * t : 4 * t * SP + 16 * q];
    }
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int j = 0; j < (LOWER ? i + 1 : NB); ++j) acc[i][j] = Mfma<T>::mma(a[i], b[j], acc[i][j]);
  }
  mfma_settle<T>();
}

// acc(c, j) -= sum_k y(k, c) B(k, j) for row tiles q0 .. q1 - 1: the right-hand
// sides y from global memory.
template <typename T, int K4, bool EX, bool BT, int q0, int q1>
__device__ __forceinline__ void staged_mma_rhs(WideAcc<T, K4>& acc, const T* y, const T* Bb, int n, int m) {
  using Sh = WideShape<T, K4, EX>;
  constexpr int NB = Sh::NB, SP = Sh::SP;
  const int r = lane_id() & 15, g = lane_id() >> 4;
  const T* b0 = Bb + (BT ? r * SP + g : g * SP + r);
#pragma unroll
  for (int t = 0; t < K4; ++t) {
    T b[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) b[j] = b0[BT ? 16 * j * SP + 4 * t : 4 * t * SP + 16 * j];
#pragma unroll
    for (int q = q0; q < q1; ++q) {
      const T a = -ldg(y, min(4 * t + g, n - 1) * m + min(16 * q + r, m - 1));
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[q][j] = Mfma<T>::mma(a, b[j], acc[q][j]);
    }
  }
  mfma_settle<T>();
}

// Where a wavefront's finished columns go: rows of a block (0: L_k, 1: R_k), or
// columns of a block or of the right-hand sides (2: Lc_k, 3: y_k).
template <typename T>
struct WideOut {
  T* to;
  int ld;  // row length of `to`
  int w, rows;
};

// Panel kb and those behind it.  acc: this wavefront's payload rows, X its
// column tile (wavefront 0: two, used in turn).
template <typename T, int K4, bool EX, int kb = 0>
__device__ __forceinline__ void wide_panels(WideAcc<T, K4>& acc, T* lds,
                                            const WideOut<T>& out, int n) {
  using Sh = WideShape<T, K4, EX>;
  constexpr int NB = Sh::NB, XP = Sh::XP;
  constexpr bool last = kb == NB - 1;
  constexpr int C = last ? Sh::NC : 16;
  const int lane = lane_id(), r = lane & 15, g = lane >> 4, w = out.w;
  T* const X0 = lds + (kb & 1) * Sh::kX;
  T* const X = w == 0 ? X0 : lds + (1 + w) * Sh::kX;
  T* const D = lds + 5 * Sh::kX;  // U_kk
  const T* const Z = D + 16 * XP;
  const bool own = w == 0, has = lane < out.rows, id = own && g == kb;
  if (out.rows > 0) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e) X[(16 * q + Mfma<T>::row(lane, e)) * XP + r] = acc[q][kb][e];
  }
  __syncthreads();
  T u[16], p[1][16];
  if (out.rows > 0) {
    run_panel<T, 1, C>(u, p, X0 + (16 * kb + r) * XP, id || !has ? Z + 15 - r : X + lane * XP);
    // (other wavefronts may still read the diagonal tile: its rows wait)
    T* to = id ? D + r * XP : X + lane * XP;
    if (has) {
#pragma unroll
      for (int c = 0; c < C; ++c) to[c] = p[0][c];
    }
  }
  __syncthreads();
  if (out.rows > 0) {
    if constexpr (!last) {
      constexpr int NJ = NB - 1 - kb;
      T b[NJ][4], a[4][4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) b[j][t] = X0[(16 * (kb + 1 + j) + r) * XP + 4 * t + g];
#pragma unroll
        for (int q = 0; q < 4; ++q) a[q][t] = -(own && q == kb ? D + r * XP : X + (16 * q + r) * XP)[4 * t + g];
      }
      // wavefront 0: U's row tile kb starts here (its accumulators took part in
      // the updates of the row tile they do not belong to)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[kb][kb + 1 + j][e] = own ? T(0) : acc[kb][kb + 1 + j][e];
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) acc[q][kb + 1 + j] = Mfma<T>::mma(a[q][t], b[j][t], acc[q][kb + 1 + j]);
    }
    if (w >= 2) {
      if (has) {
#pragma unroll
        for (int c = 0; c < C; ++c)
          if (EX || 16 * kb + c < n) stg(out.to, (16 * kb + c) * out.ld + lane, p[0][c]);
      }
    } else {
      if (id) {  // L_kk with U_kk above its diagonal
#pragma unroll
        for (int c = 0; c < C; ++c) X0[(16 * kb + r) * XP + c] = (c <= r) ? u[c] : p[0][c];
      }
      wave_lds_order();
#pragma unroll
      for (int q = 0; q < NB; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int row = 16 * q + Mfma<T>::row(lane, e), col = 16 * kb + r;
          const T v = X[row * XP + r];
          if (row < n && col < n) stg(out.to, row * n + col, v);
        }
    }
    mfma_settle<T>();
  }
  if constexpr (!last) wide_panels<T, K4, EX, kb + 1>(acc, lds, out, n);
}

template <typename T, int K4, bool EX>
__global__ __launch_bounds__(kWideThreads) void k_wide_up(SmallArgs<T> A, int l) {
  using Sh = WideShape<T, K4, EX>;
  constexpr int NB = Sh::NB, SP = Sh::SP;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T* const lds = reinterpret_cast<T*>(smem_raw);
  SmallSys<T> Q;
  int task;
  if (!small_sys(A, Q, task)) return;
  const int w = wave_uniform(), lane = lane_id(), r = lane & 15;
  const int N = Q.N, n = EX ? 4 * K4 : Q.n, m = Q.m, nn = n * n, nm = n * m;
  const int s = 1 << l, h = s >> 1, dim = (N + s) / (2 * s);
  const bool node = task < dim;
  const int k = node ? s - 1 + 2 * s * task : 2 * s * (task - dim + 1) - 1;
  const int lp = l > 0 ? l - 1 : 0;
  const int offp = seg_offset(N, lp), off = l > 0 ? offp + (N >> lp) - 1 : 0;
  const bool hasR = node && k + s < N, hasC = node && k >= s;
  T* const Rk = Q.E + (size_t)(off + (k >> l)) * nn;
  T* const Lck = Q.E + (size_t)(off + ((k - s) >> l)) * nn;
  T* const Lk = Q.L + (size_t)k * nn;
  const T* const Lin = (l <= 1 ? Q.Lin : Q.L) + (size_t)k * nn;  // first read at level 0 or 1
  T* const yk = Q.x != nullptr ? Q.x + (size_t)k * nm : nullptr;
  // staged blocks: R_{k-h}, Lc_{k+h}, Lc_{k-h}, R_{k+h}; level 0: Lc_k
  T* const B0 = lds;
  T* const B1 = B0 + Sh::kBlock;
  T* const B2 = B1 + Sh::kBlock;
  T* const B3 = B2 + Sh::kBlock;
  const bool up = l > 0, right = up && k + h < N;

  {
    Staged<T, K4, EX> s0, s1, s2, s3;
    if (up) {
      s0.load(Q.E + (size_t)(offp + ((k - h) >> lp)) * nn, n, w);
      if (right) s1.load(Q.E + (size_t)(offp + (k >> lp)) * nn, n, w);
      if (hasC) s2.load(Q.E + (size_t)(offp + ((k - s) >> lp)) * nn, n, w);
      if (hasR) s3.load(Q.E + (size_t)(offp + ((k + h) >> lp)) * nn, n, w);
      s0.store(B0, n, w);
      if (right) s1.store(B1, n, w);
      if (hasC) s2.store(B2, n, w);
      if (hasR) s3.store(B3, n, w);
    } else if (hasC) {
      s2.load(Q.Ein + (Lck - Q.E), n, w);
      s2.store(B0, n, w);
    }
  }
  __syncthreads();
  WideAcc<T, K4> acc;
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[q][j] = acc_zero<T>();
  if (w == 0) {
    // (the block itself arrives under the products)
    typename Mfma<T>::acc_t d[NB * (NB + 1) / 2];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int j = 0; j <= i; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          d[i * (i + 1) / 2 + j][e] =
              ldg(Lin, min(16 * i + Mfma<T>::row(lane, e), n - 1) * n + min(16 * j + r, n - 1));
    if (up) staged_mma<T, K4, EX, false, true, true>(acc, B0, B0);
    if (right) staged_mma<T, K4, EX, true, false, true>(acc, B1, B1);
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int j = 0; j <= i; ++j) {
        acc[i][j] += d[i * (i + 1) / 2 + j];
        if (!EX || 4 * K4 < Sh::NP) {  // identity padding
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int row = 16 * i + Mfma<T>::row(lane, e), col = 16 * j + r;
            acc[i][j][e] = (row < n && col < n) ? acc[i][j][e] : ((row == col) ? T(1) : T(0));
          }
        }
      }
  } else if (w == 1) {
    if (hasR) {
      if (up) {
        staged_mma<T, K4, EX, false, false, false>(acc, B3, B1);  // R_{k+h} Lc_{k+h}
      } else {
        const T* M = Q.Ein + (Rk - Q.E);
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
          for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              acc[i][j][e] = ldg(M, min(16 * i + Mfma<T>::row(lane, e), n - 1) * n + min(16 * j + r, n - 1));
      }
    }
  } else if (w == 2) {
    if (hasC) {
      if (up) {
        staged_mma<T, K4, EX, true, true, false>(acc, B2, B0);  // (R_{k-h} Lc_{k-h})^T
      } else {
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
          for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i][j][e] = B0[(16 * j + r) * SP + 16 * i + Mfma<T>::row(lane, e)];
      }
    }
  } else if (yk != nullptr) {
    auto columns = [&](auto q0c, auto q1c) {
      constexpr int q0 = decltype(q0c)::value, q1 = decltype(q1c)::value;
#pragma unroll
      for (int q = q0; q < q1; ++q)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            acc[q][j][e] = ldg(yk, min(16 * j + r, n - 1) * m + min(16 * q + Mfma<T>::row(lane, e), m - 1));
      if (up) staged_mma_rhs<T, K4, EX, true, q0, q1>(acc, yk - (size_t)h * nm, B0, n, m);
      if (right) staged_mma_rhs<T, K4, EX, false, q0, q1>(acc, yk + (size_t)h * nm, B1, n, m);
    };
    columns(std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{});
    if (m > 16) columns(std::integral_constant<int, 1>{}, std::integral_constant<int, 4>{});
  }

  if (!node) {
    if (w == 0) {
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j <= i; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int row = 16 * i + Mfma<T>::row(lane, e), col = 16 * j + r;
            if (col <= row && row < n) stg(Lk, row * n + col, acc[i][j][e]);
          }
    } else if (w == 3 && yk != nullptr) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int c = 16 * q + Mfma<T>::row(lane, e);
            if (c < m && 16 * j + r < n) stg(yk, (16 * j + r) * m + c, acc[q][j][e]);
          }
    }
    return;
  }
  __syncthreads();  // the staged blocks' LDS is the column tiles' from here
  T* const Z = lds + 5 * Sh::kX + 16 * Sh::XP;
  if (w == 3 && lane < 32) Z[lane] = lane == 15 ? T(1) : T(0);
  WideOut<T> out;
  out.w = w;
  out.to = w == 0 ? Lk : (w == 1 ? Rk : (w == 2 ? Lck : yk));
  out.ld = w == 3 ? m : n;
  out.rows = w == 0 ? Sh::NP : (w == 1 ? (hasR ? Sh::NP : 0) : (w == 2 ? (hasC ? n : 0) : (yk != nullptr ? m : 0)));
  wide_panels<T, K4, EX>(acc, lds, out, n);
}

// f(K4, EX as integral constants)
template <typename F>
void with_wide(int n, F f) {
  using std::integral_constant;
  const int k4 = (n + 7) / 8 * 2;
  const bool ex = n == 4 * k4;
  auto go = [&](auto k) {
    if (ex) f(k, integral_constant<bool, true>{});
    else f(k, integral_constant<bool, false>{});
  };
  if (k4 == 10) go(integral_constant<int, 10>{});
  else if (k4 == 12) go(integral_constant<int, 12>{});
  else if (k4 == 14) go(integral_constant<int, 14>{});
  else go(integral_constant<int, 16>{});
}

template <typename T>
hipError_t set_attrs() {
  hipError_t e = hipSuccess;
  for (int n = 33; n <= 64 && e == hipSuccess; ++n)
    with_wide(n, [&](auto k4, auto ex) {
      constexpr int K4 = decltype(k4)::value;
      constexpr bool EX = decltype(ex)::value;
      e = hipFuncSetAttribute((const void*)k_wide_up<T, K4, EX>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)(sizeof(T) * WideShape<T, K4, EX>::elems(4)));
    });
  return e;
}

}  // namespace

hipError_t init_wide_kernels() {
  const hipError_t e = set_attrs<float>();
  return e == hipSuccess ? set_attrs<double>() : e;
}

template <typename T>
hipError_t wide_up_level(T* L, T* E, T* x, const uint8_t* mask, int B, int N, int n, int m, int l, hipStream_t st,
                         const T* Lsrc, const T* Esrc) {
  if (n <= kSmallN || n > kSmallUpN) return hipErrorInvalidValue;
  if (B <= 0) return hipSuccess;
  const Level lv = level_info(N, l);
  const int tasks = lv.dim + (l > 0 ? N / (2 * lv.s) : 0);
  kt_begin(kKcPotrf, st);
  with_wide(n, [&](auto k4, auto ex) {
    constexpr int K4 = decltype(k4)::value;
    constexpr bool EX = decltype(ex)::value;
    const size_t lds = sizeof(T) * (l > 0 ? WideShape<T, K4, EX>::elems(4) : WideShape<T, K4, EX>::elems(1));
    hipLaunchKernelGGL((k_wide_up<T, K4, EX>), dim3(tasks, B), dim3(kWideThreads), lds, st,
                       regular_args(L, E, x, mask, N, n, m, Lsrc, Esrc), l);
  });
  kt_end(kKcPotrf, st);
  return hipGetLastError();
}

template hipError_t wide_up_level<float>(float*, float*, float*, const uint8_t*, int, int, int, int, int, hipStream_t,
                                         const float*, const float*);
template hipError_t wide_up_level<double>(double*, double*, double*, const uint8_t*, int, int, int, int, int,
                                          hipStream_t, const double*, const double*);

}  // namespace socu
