// Cholesky factor and inverse of diagonal blocks up to n = 128, one workgroup
// of up to four wavefronts per block:
//   k_potrf_blk  A = L L^T (reference: potrf_blocked, socu/blas/potrf.py:97-119),
//                L into the lower triangle and U = L^-T into the strict upper
//                triangle, which is not part of the factor (the reference only
//                ever reads tril(L));
//   k_trtri_blk  the same U from tril(L) alone, for solves whose factor may come
//                from anywhere (potrf.py:101-103).
//
// The panel factor of nd_panel.h with one payload row per lane: wavefront w owns
// the 16-row tiles w and w + 4, and keeps their unfinished columns in registers,
// as MFMA accumulators.  A row tile i is rows of A until its own panel i, from
// where on it is rows of U (the identity, transformed).  Per panel of 16
// columns: the column tile goes through LDS into the one-row-per-lane form,
// every wavefront factors the 16x16 diagonal tile itself and transforms its
// rows with it, the result goes through LDS into the operand form, and MFMAs
// update the column tiles to the right.
//
// What bounds it: one workgroup's serial work.  FP64, n = 128: 66k cycles (28 us),
// of which 4k the load (one compute unit's misses), 17k the pivot chains (2.1k
// each), 20k the MFMAs (224 per wavefront; they share the FP64 units with the
// chains' multiply-adds: issued between a chain's steps they lengthened it by
// their own time) and the rest the four LDS passes and two barriers per panel.
// With 32x32 tiles the kernel took the same at n = 128 but worked on whole tiles
// below it: FP64 factor_and_solve n=80 N=200 512 -> 382 us, n=100 N=256 m=4
// 938 -> 664 us (sweeps included), FP32 n=112 N=200 514 -> 391 us.  The inverses
// alone: n=100, 200 blocks 42 -> 23 us, n=34, 128 blocks 18 -> 6 us.
#include <stdlib.h>

#include <hip/hip_ext.h>

#include "../../include/socu_hip.h"
#include "nd_common.h"
#include "nd_internal.h"
#include "nd_small.h"
#include "nd_tile.h"

namespace socu {

namespace {

constexpr int kXP = 18;  // pitch of a column tile: rows in pairs of entries, no bank conflicts

template <int NB>
struct TriShape {
  static constexpr int Q = NB > 4 ? 2 : 1;   // row tiles per wavefront
  static constexpr int W = NB < 4 ? NB : 4;  // wavefronts
  static constexpr int NP = 16 * W * Q;      // rows (those behind the block: zeros)
  static constexpr int kThreadsT = 64 * W;
  static constexpr int CT = NP * kXP;
  // two column tiles, used in turn; U_kk; the identity
  static constexpr int elems = 2 * CT + 2 * 16 * kXP;
};

template <typename T, int NB>
using TriAcc = typename Mfma<T>::acc_t[TriShape<NB>::Q][NB];

// A payload row through a given triangle: p <- p L^-T, u holding row
// (lane % 16) of L, rinv its 1 / L[r][r].
template <typename T>
__device__ __forceinline__ void panel16_given(T (&u)[16], T (&p)[16], T rinv) {
  pin_reg(rinv);
  __builtin_amdgcn_sched_barrier(0);
  wait_states<2>();
  static_for<16>([&](auto kc) {
    constexpr int k = decltype(kc)::value;
    p[k] *= bcast_row<k>(rinv);
    static_for<15 - k>([&](auto qc) {
      constexpr int q = k + 1 + decltype(qc)::value;
      fnma_row<q>(p[q], u[k], p[k]);
    });
  });
}

// 16 consecutive entries (aligned to two).
template <typename T>
__device__ __forceinline__ void read16(T (&v)[16], const T* row) {
  typedef T v2 __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const v2 d = reinterpret_cast<const v2*>(row)[c];
    v[2 * c] = d.x;
    v[2 * c + 1] = d.y;
  }
}
template <typename T>
__device__ __forceinline__ void write16(T* row, const T (&v)[16]) {
  typedef T v2 __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int c = 0; c < 8; ++c) reinterpret_cast<v2*>(row)[c] = v2{v[2 * c], v[2 * c + 1]};
}
// MFMA operand: lane group g takes k = 4 g + t in MFMA t.
template <typename T>
__device__ __forceinline__ void read4(T (&v)[4], const T* row, int g) {
  typedef T v2 __attribute__((ext_vector_type(2)));
  const v2* const q = reinterpret_cast<const v2*>(row + 4 * g);
  const v2 d0 = q[0], d1 = q[1];
  v[0] = d0.x;
  v[1] = d0.y;
  v[2] = d1.x;
  v[3] = d1.y;
}

// Column tile kb, finished, to memory: read from LDS before the next panel and
// stored behind it.
template <typename T, typename TS, int NB, int kb>
struct TriStore {
  static constexpr int Q = TriShape<NB>::Q;
  T v[Q][4];
  __device__ __forceinline__ void read(const T* X) {
    const int lane = lane_id(), w = wave_uniform();
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[q][e] = X[(16 * (w + 4 * q) + 4 * e + (lane >> 4)) * kXP + (lane & 15)];
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e) pin_reg(v[q][e]);
  }
  __device__ __forceinline__ void write(TS* out, int ld, int n) {
    const int lane = lane_id(), w = wave_uniform();
    const int col = 16 * kb + (lane & 15);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int row = 16 * (w + 4 * q) + (lane >> 4);
      if (16 * (w + 4 * q) + 16 <= n && 16 * kb + 16 <= n) {
#pragma unroll
        for (int e = 0; e < 4; ++e) stg(out, (row + 4 * e) * ld + col, (TS)v[q][e]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (row + 4 * e < n && col < n) stg(out, (row + 4 * e) * ld + col, (TS)v[q][e]);
      }
    }
  }
};

// Panel kb and those behind it.
template <typename T, typename TS, int NB, bool GIVEN, int kb = 0>
__device__ __forceinline__ void tri_panels(TriAcc<T, NB>& acc, T* lds, TS* out, int ld, int n) {
  using Sh = TriShape<NB>;
  constexpr int Q = Sh::Q, XP = kXP;
  constexpr bool last = kb == NB - 1;
  const int lane = lane_id(), r = lane & 15, g = lane >> 4, w = wave_uniform();
  T* const X = lds + (kb & 1) * Sh::CT;
  T* const D = lds + 2 * Sh::CT;
  const T* const I = D + 16 * XP;
#pragma unroll
  for (int q = 0; q < Q; ++q)
#pragma unroll
    for (int e = 0; e < 4; ++e) X[(16 * (w + 4 * q) + Mfma<T>::row(lane, e)) * XP + r] = acc[q][kb][e];
  __syncthreads();
  const int it = w + 4 * (g & (Q - 1));  // this lane's row: r of tile it
  const bool id = it == kb, has = g < Q && (!GIVEN || it <= kb);
  T* const xrow = X + (16 * it + r) * XP;
  T u[16], p[1][16];
  const T* const urow = X + (16 * kb + r) * XP;
  TriStore<T, TS, NB, kb - 1> st;
  if constexpr (kb > 0) st.read(lds + ((kb - 1) & 1) * Sh::CT);
  read16(u, urow);
  read16(p[0], id ? I + r * XP : xrow);
#pragma unroll
  for (int c = 0; c < 16; ++c) {
    pin_reg(u[c]);
    pin_reg(p[0][c]);
  }
  if constexpr (GIVEN) panel16_given(u, p[0], T(1) / urow[r]);
  else panel16<T, 1, 16>(u, p);
  if constexpr (kb > 0) st.write(out, ld, n);
  // (other wavefronts may still read the diagonal tile: its rows wait)
  if (has) write16(id ? D + r * XP : xrow, p[0]);
  __syncthreads();
  if constexpr (!last) {
    constexpr int NJ = NB - 1 - kb;
    T a[Q][4], b[NJ][4];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int i = w + 4 * q;
      read4(a[q], (i == kb ? D : X + 16 * i * XP) + r * XP, g);
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) read4(b[j], X + (16 * (kb + 1 + j) + r) * XP, g);
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int t = 0; t < 4; ++t) a[q][t] = (GIVEN && w + 4 * q > kb) ? T(0) : -a[q][t];
    // Every row takes every column to the right, a row of A also those behind its
    // own, which do not count: the wavefronts wait for the one with the most
    // updates (50 tiles to 56 over the 8 panels of n = 128), and a branch per tile
    // costs more, in accumulators moved about.  Rows of U start from zero here.
    if (w == kb % 4) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[kb / 4][kb + 1 + j] = acc_zero<T>();
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int q = 0; q < Q; ++q) acc[q][kb + 1 + j] = Mfma<T>::mma(a[q][t], b[j][t], acc[q][kb + 1 + j]);
  }
  if (id && g < Q) {  // L_kk with U_kk above its diagonal
#pragma unroll
    for (int c = 0; c < 16; ++c) u[c] = (c <= r) ? u[c] : p[0][c];
    write16(xrow, u);
  }
  mfma_settle<T>();
  if constexpr (last) {
    wave_lds_order();
    TriStore<T, TS, NB, kb> fin;
    fin.read(X);
    fin.write(out, ld, n);
  } else {
    tri_panels<T, TS, NB, GIVEN, kb + 1>(acc, lds, out, ld, n);
  }
}

// in (n x n, row length ld; its lower triangle is read) -> out.
template <typename T, typename TS, int NB, bool GIVEN>
__device__ __forceinline__ void tri_block(T* lds, const TS* in, TS* out, int ld, int n) {
  using Sh = TriShape<NB>;
  constexpr int Q = Sh::Q;
  const int lane = lane_id(), r = lane & 15, w = wave_uniform();
  TS v[Q][NB][4];
#pragma unroll
  for (int q = 0; q < Q; ++q)
#pragma unroll
    for (int j = 0; j < (q < Q - 1 ? 4 : NB); ++j)  // (tile row w + 4 q has columns 0 .. w + 4 q)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (j <= w + 4 * q)
          v[q][j][e] = ldg(in, min(16 * (w + 4 * q) + Mfma<T>::row(lane, e), n - 1) * ld + min(16 * j + r, n - 1));
  T* const I = lds + 2 * Sh::CT + 16 * kXP;
  for (int c = threadIdx.x; c < 256; c += Sh::kThreadsT) I[(c >> 4) * kXP + (c & 15)] = (c >> 4) == (c & 15) ? T(1) : T(0);
  TriAcc<T, NB> acc;
#pragma unroll
  for (int q = 0; q < Q; ++q)
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      acc[q][j] = acc_zero<T>();
      if (j < (q < Q - 1 ? 4 : NB)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          pin_reg(v[q][j][e]);
          // identity padding; above the diagonal 0
          const int row = 16 * (w + 4 * q) + Mfma<T>::row(lane, e), col = 16 * j + r;
          acc[q][j][e] = (row < n && col <= row) ? (T)v[q][j][e] : ((row == col) ? T(1) : T(0));
        }
      }
    }
  tri_panels<T, TS, NB, GIVEN>(acc, lds, out, ld, n);
}

// Block (r0, r0) of size nb of the nodes i = s-1+2st's diagonal blocks (grid
// (nodes, B)); Lsrc: where it is read (NULL: in place).
template <typename TS, typename T, int NB>
__global__ __launch_bounds__(TriShape<NB>::kThreadsT) void k_potrf_blk(TS* L, const uint8_t* __restrict__ mask, int N,
                                                                      int n, int s, const TS* Lsrc, int r0, int nb) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T* const lds = reinterpret_cast<T*>(smem_raw);
  const int b = blockIdx.y;
  if (masked_out(mask, b)) return;
  const int i = s - 1 + 2 * s * blockIdx.x;
  const size_t o = ((size_t)b * N + i) * n * n + (size_t)r0 * (n + 1);
  tri_block<T, TS, NB, false>(lds, (Lsrc != nullptr ? Lsrc : L) + o, L + o, n, nb);
}

// The same block of every diagonal block: W <- tril(L) and U (grid (N, B)).
template <typename T, int NB>
__global__ __launch_bounds__(TriShape<NB>::kThreadsT) void k_trtri_blk(const T* __restrict__ L, T* __restrict__ W,
                                                                      const uint8_t* __restrict__ mask, int N, int n,
                                                                      int r0, int nb) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T* const lds = reinterpret_cast<T*>(smem_raw);
  const int b = blockIdx.y;
  if (masked_out(mask, b)) return;
  const size_t o = ((size_t)b * N + blockIdx.x) * n * n + (size_t)r0 * (n + 1);
  tri_block<T, T, NB, true>(lds, L + o, W + o, n, nb);
}

template <typename F>
void with_tiles(int nb, F f) {
  switch ((nb + 15) / 16) {
    case 1: f(std::integral_constant<int, 1>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 3: f(std::integral_constant<int, 3>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 5: f(std::integral_constant<int, 5>{}); break;
    case 6: f(std::integral_constant<int, 6>{}); break;
    case 7: f(std::integral_constant<int, 7>{}); break;
    default: f(std::integral_constant<int, 8>{}); break;
  }
}

template <typename TS, typename T>
hipError_t launch_potrf(TS* L, const uint8_t* mask, int B, int N, int n, int lidx, const TS* Lsrc, int r0, int nb,
                        hipStream_t st) {
  const Level lv = level_info(N, lidx);
  if (nb < 1 || nb > kMaxN || r0 < 0 || r0 + nb > n) return hipErrorInvalidValue;
  if (lv.dim <= 0 || B <= 0) return hipSuccess;
  with_tiles(nb, [&](auto tiles) {
    constexpr int NB = decltype(tiles)::value;
    const dim3 grid(lv.dim, B), block(TriShape<NB>::kThreadsT);
    const size_t lds = sizeof(T) * TriShape<NB>::elems;
    // under socu_profile_op the launch itself records its start and end
    // (events of hipExtLaunchKernel: the kernel's own execution interval)
    hipEvent_t ea = nullptr, eb = nullptr;
    if (kt_kernel_events(kKcPotrf, &ea, &eb))
      hipExtLaunchKernelGGL((k_potrf_blk<TS, T, NB>), grid, block, lds, st, ea, eb, 0, L, mask, N, n, lv.s, Lsrc, r0, nb);
    else
      hipLaunchKernelGGL((k_potrf_blk<TS, T, NB>), grid, block, lds, st, L, mask, N, n, lv.s, Lsrc, r0, nb);
  });
  return hipGetLastError();
}

template <typename F>
hipError_t set_attr(F* f, size_t lds) {
  return hipFuncSetAttribute((const void*)f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
}

}  // namespace

hipError_t init_potrf_kernels() {
  hipError_t e = hipSuccess;
  for (int nb = 1; nb <= kMaxN && e == hipSuccess; nb += 16)
    with_tiles(nb, [&](auto tiles) {
      constexpr int NB = decltype(tiles)::value;
      constexpr size_t lds = TriShape<NB>::elems;
      e = set_attr(k_potrf_blk<float, float, NB>, sizeof(float) * lds);
      if (e == hipSuccess) e = set_attr(k_potrf_blk<float, double, NB>, sizeof(double) * lds);
      if (e == hipSuccess) e = set_attr(k_potrf_blk<double, double, NB>, sizeof(double) * lds);
      if (e == hipSuccess) e = set_attr(k_trtri_blk<float, NB>, sizeof(float) * lds);
      if (e == hipSuccess) e = set_attr(k_trtri_blk<double, NB>, sizeof(double) * lds);
    });
  return e;
}

template <typename T>
hipError_t potrf_level(T* L, const uint8_t* mask, int B, int N, int n, int lidx, bool f64, const T* Lsrc, int r0,
                       int nb, hipStream_t st) {
  if (f64) return launch_potrf<T, double>(L, mask, B, N, n, lidx, Lsrc, r0, nb, st);
  return launch_potrf<T, T>(L, mask, B, N, n, lidx, Lsrc, r0, nb, st);
}

template <typename T>
hipError_t trtri_blocks(const T* L, T* W, const uint8_t* mask, int B, int N, int n, int r0, int nb, hipStream_t st) {
  if (nb < 1 || nb > kMaxN || r0 < 0 || r0 + nb > n) return hipErrorInvalidValue;
  if (B <= 0) return hipSuccess;
  with_tiles(nb, [&](auto tiles) {
    constexpr int NB = decltype(tiles)::value;
    hipLaunchKernelGGL((k_trtri_blk<T, NB>), dim3(N, B), dim3(TriShape<NB>::kThreadsT),
                       sizeof(T) * TriShape<NB>::elems, st, L, W, mask, N, n, r0, nb);
  });
  return hipGetLastError();
}

template hipError_t potrf_level<float>(float*, const uint8_t*, int, int, int, int, bool, const float*, int, int,
                                       hipStream_t);
template hipError_t potrf_level<double>(double*, const uint8_t*, int, int, int, int, bool, const double*, int, int,
                                        hipStream_t);
template hipError_t trtri_blocks<float>(const float*, float*, const uint8_t*, int, int, int, int, int, hipStream_t);
template hipError_t trtri_blocks<double>(const double*, double*, const uint8_t*, int, int, int, int, int, hipStream_t);

}  // namespace socu
