// Blocked ND kernels for block size n <= 128 on gfx950: blocks are padded to
// NP = 32*NB (NB = ceil(n/32)) inside LDS/registers only; HBM accesses stay
// within the n x n blocks.  One or two kernel launches per phase per level; no
// atomics, so results are bitwise reproducible.
//
//   k_potrf_blk  (nd_potrf.hip) L_i and its inverse's transpose.
//   k_large_panel (nd_large.hip) R <- R U, Lc <- U^T Lc with the stored inverse
//                (replaces trsm_rltn / trsm_llnn, trsm.py:94-120, :202-228).
//   k_schur_blk  one workgroup per 64x64 output tile, MFMA, owner computes:
//                L_j -= R R^T + Lc^T Lc,  F -= R Lc (syrk.py, gemm.py).
// (The sweeps: nd_small.hip, nd_steps.hip, nd_large.hip.)
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include <hip/hip_ext.h>

#include "nd_common.h"
#include "nd_internal.h"
#include "nd_tile.h"

namespace socu {

// NF != 0 instantiates the kernels for a fixed block size n == NF (a multiple
// of 32), so that all index arithmetic is compile-time; NF == 0 is the
// general (padded) version.

// ---------------------------------------------------------------------------
// Schur-complement updates, 64x64 output tiles on MFMA
// ---------------------------------------------------------------------------
constexpr int kSTile = 64;
constexpr int kSK = 32;
constexpr int kSP = kSTile + 1;

enum { kABt = 0, kAtB = 1, kAB = 2 };

// One K-chunk of both operands of a 64x64 tile product, held in registers
// between the global loads and the LDS stores so that the next chunk's loads
// are in flight while the current chunk is multiplied.
// As[kk][a] = A(r0+a, k0+kk), Bs[kk][a] = B(k0+kk, c0+a), zero outside n.
constexpr int kSPer = kSTile * kSK / kThreads;  // elements per thread per operand

template <typename T>
struct Chunk64 {
  T a[kSPer];
  T b[kSPer];
};

template <typename T>
__device__ __forceinline__ void load_chunk64(Chunk64<T>& ch, const T* __restrict__ Am, const T* __restrict__ Bm,
                                             int form, int n, int r0, int c0, int k0) {
#pragma unroll
  for (int e = 0; e < kSPer; ++e) {
    const int idx = threadIdx.x + e * kThreads;
    const int a = idx / kSK, kk = idx - a * kSK, k = k0 + kk;                // k fastest: row reads
    const int kk2 = idx / kSTile, a2 = idx - kk2 * kSTile, k2 = k0 + kk2;  // a fastest: column reads
    // unconditional loads from clamped addresses, then select
    const int ra = min(r0 + a, n - 1), ca = min(c0 + a, n - 1), kc = min(k, n - 1);
    const int ra2 = min(r0 + a2, n - 1), ca2 = min(c0 + a2, n - 1), kc2 = min(k2, n - 1);
    const bool va = r0 + a < n && k < n, vb = c0 + a < n && k < n;
    const bool va2 = r0 + a2 < n && k2 < n, vb2 = c0 + a2 < n && k2 < n;
    if (form == kABt) {
      const T x = Am[(size_t)ra * n + kc], y = Bm[(size_t)ca * n + kc];
      ch.a[e] = va ? x : T(0);
      ch.b[e] = vb ? y : T(0);
    } else if (form == kAtB) {
      const T x = Am[(size_t)kc2 * n + ra2], y = Bm[(size_t)kc2 * n + ca2];
      ch.a[e] = va2 ? x : T(0);
      ch.b[e] = vb2 ? y : T(0);
    } else {
      const T x = Am[(size_t)ra * n + kc], y = Bm[(size_t)kc2 * n + ca2];
      ch.a[e] = va ? x : T(0);
      ch.b[e] = vb2 ? y : T(0);
    }
  }
}

template <typename T>
__device__ __forceinline__ void store_chunk64(const Chunk64<T>& ch, T* As, T* Bs, int form) {
#pragma unroll
  for (int e = 0; e < kSPer; ++e) {
    const int idx = threadIdx.x + e * kThreads;
    const int a = idx / kSK, kk = idx - a * kSK;
    const int kk2 = idx / kSTile, a2 = idx - kk2 * kSTile;
    if (form == kAtB) As[kk2 * kSP + a2] = ch.a[e];
    else As[kk * kSP + a] = ch.a[e];
    if (form == kABt) Bs[kk * kSP + a] = ch.b[e];
    else Bs[kk2 * kSP + a2] = ch.b[e];
  }
}

// Sequence of up to two products over K chunks: acc += sum_p A_p B_p (BF:
// on BF16 MFMA, float storage).
template <typename T, bool BF>
__device__ __forceinline__ void products64(typename Mfma<T>::acc_t acc[2][2], bool active, int np, const T* const* Am,
                                           const T* const* Bm, const int* form, int n, int r0, int c0, T* As, T* Bs) {
  const int wave = wave_id();
  const int wi = wave >> 1, wj = wave & 1;
  const int nk = (n + kSK - 1) / kSK;
  const int total = np * nk;
  Chunk64<T> ch;
  load_chunk64<T>(ch, Am[0], Bm[0], form[0], n, r0, c0, 0);
  for (int q = 0; q < total; ++q) {
    const int p = q / nk;
    __syncthreads();
    store_chunk64<T>(ch, As, Bs, form[p]);
    __syncthreads();
    if (q + 1 < total) {
      const int p1 = (q + 1) / nk, k1 = ((q + 1) - p1 * nk) * kSK;
      load_chunk64<T>(ch, Am[p1], Bm[p1], form[p1], n, r0, c0, k1);
    }
    if (active) schur_gemm<T, BF>(acc, As + 32 * wi, 1, kSP, Bs + 32 * wj, kSP, 1, kSK);
  }
}

// Workgroups are handed to the eight XCDs round-robin (XCD = workgroup index
// mod 8, gridDim.x a multiple of 8), and each XCD has its own L2.  Tasks are
// numbered group-major -- group g: the output tiles of target g, then those
// of fill-in g, which share E blocks 2g+1 (and read 2g, 2g+2) -- and XCD x
// takes the contiguous range [x * per, (x + 1) * per) of that order, so the
// tiles that re-read one operand block run on one XCD at about the same
// time.  Slots past the last task (and the missing fill-in of the last
// group) return at once.
__host__ __device__ constexpr int schur_blk_groups(int nT, int nF) { return nT > nF ? nT : nF; }
__host__ __device__ constexpr int schur_blk_per_xcd(int nT, int nF, int ntile) {
  return (schur_blk_groups(nT, nF) * (ntile * (ntile + 1) / 2 + ntile * ntile) + 7) / 8;
}

template <typename T, int NF, bool BF = false>
__global__ __launch_bounds__(kThreads) void k_schur_blk(T* __restrict__ L, T* __restrict__ E,
                                                       const uint8_t* __restrict__ mask, int N, int n_, int nE, int s,
                                                       int off, int next_off, int nT, int nF, int ntile,
                                                       const T* __restrict__ Lsrc) {
  const int n = NF ? NF : n_;
  const int b = blockIdx.y;
  if (masked_out(mask, b)) return;
  __shared__ T As[kSK * kSP];
  __shared__ T Bs[kSK * kSP];
  const int ntri = ntile * (ntile + 1) / 2;
  const int gs = ntri + ntile * ntile;
  int task;
  bool target;
  {
    const int per = schur_blk_per_xcd(nT, nF, ntile);
    const int lg = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    const int g = lg / gs, q = lg - g * gs;
    target = q < ntri;
    if (target ? g >= nT : g >= nF) return;
    task = target ? g * ntri + q : nT * ntri + g * ntile * ntile + (q - ntri);
  }
  const size_t nn = (size_t)n * n;
  T* Eb = E + (size_t)b * nE * nn;
  const int wave = wave_id();
  const int wi = wave >> 1, wj = wave & 1;
  typename Mfma<T>::acc_t acc[2][2] = {{acc_zero<T>(), acc_zero<T>()}, {acc_zero<T>(), acc_zero<T>()}};
  T* C;
  int tr, tc;
  bool active = true;
  if (target) {
    const int u = task / ntri;
    int q = task - u * ntri;
    tr = 0;
    while (q > tr) { q -= tr + 1; ++tr; }
    tc = q;
    active = !(tr == tc && wi < wj);  // upper 32x32 quarter of a diagonal tile
    const int j = 2 * s * (u + 1) - 1;
    C = L + ((size_t)b * N + j) * nn;
    const T* R = Eb + (size_t)(off + (j - s) / s) * nn;
    const T* Lc = (j + s < N) ? Eb + (size_t)(off + j / s) * nn : R;
    const T* Am[2] = {R, Lc};
    const int form[2] = {kABt, kAtB};
    products64<T, BF>(acc, active, (j + s < N) ? 2 : 1, Am, Am, form, n, tr * kSTile, tc * kSTile, As, Bs);
  } else {
    task -= nT * ntri;
    const int f = task / (ntile * ntile);
    const int q = task - f * ntile * ntile;
    tr = q / ntile;
    tc = q - tr * ntile;
    const int i = s - 1 + 2 * s * (f + 1);
    const T* R = Eb + (size_t)(off + i / s) * nn;
    const T* Lc = Eb + (size_t)(off + (i - s) / s) * nn;
    C = Eb + (size_t)(next_off + (i - s) / (2 * s)) * nn;
    const T* Am[1] = {R};
    const T* Bm[1] = {Lc};
    const int form[1] = {kAB};
    products64<T, BF>(acc, active, 1, Am, Bm, form, n, tr * kSTile, tc * kSTile, As, Bs);
  }
  if (!active) return;
  const int rb = tr * kSTile + 32 * wi, cb = tc * kSTile + 32 * wj;
  if (target) {
    // (out-of-place: the target is read from Lsrc, same layout)
    const T* Cin = (Lsrc != nullptr) ? Lsrc + (C - L) : C;
    acc_foreach<T>(acc, [&](int r, int c, T v) {
      const int rr = rb + r, cc = cb + c;
      if (rr < n && cc < n) C[(size_t)rr * n + cc] = Cin[(size_t)rr * n + cc] - v;
    });
  } else {
    // the fill-in block receives its only update here: F = -R Lc, whatever
    // it held on entry (the reference's F -= R Lc on a zeroed block)
    acc_foreach<T>(acc, [&](int r, int c, T v) {
      const int rr = rb + r, cc = cb + c;
      if (rr < n && cc < n) C[(size_t)rr * n + cc] = -v;
    });
  }
}

// ---------------------------------------------------------------------------
// BF16 Schur products for levels with few nodes, and those of FP32 blocks of
// 16 < n <= 32.  k_schur_blk walks K in chunks, one global round trip per chunk,
// which at the upper levels (a handful of tiles) is the whole cost.  Here a task is
// a 32x32 output tile (4x more tasks) and issues every load it needs at once: the 32-wide panels
// of its operands (all of K) and its own C values, then one LDS staging and
// the MFMA products.  Panels are kept as P[i][k] (pitch NP + 1): row panels
// are 32 rows of a block, column panels 32 of its columns, transposed.
// ---------------------------------------------------------------------------
// four panels of 32 x (NP+1)
template <typename T, int NB>
constexpr size_t schur_small_lds() {
  return sizeof(T) * 4 * 32 * (size_t)(32 * NB + 1);
}

template <typename T, int NB>
__device__ __forceinline__ void panel_load(T* v, const T* __restrict__ M, bool cols, int i0, int n) {
  constexpr int NP = 32 * NB;
  constexpr int PE = 32 * NP / kThreads;
#pragma unroll
  for (int e = 0; e < PE; ++e) {
    const int idx = threadIdx.x + e * kThreads;
    int i, k;
    if (!cols) {  // row panel: contiguous along k
      i = idx / NP;
      k = idx - i * NP;
    } else {      // column panel: 32 contiguous entries of each row k
      k = idx >> 5;
      i = idx & 31;
    }
    const int rr = cols ? k : i0 + i, cc = cols ? i0 + i : k;
    v[e] = M[min(rr, n - 1) * n + min(cc, n - 1)];
  }
}

template <typename T, int NB>
__device__ __forceinline__ void panel_store(T* P, const T* v, bool cols, int i0, int n) {
  constexpr int NP = 32 * NB;
  constexpr int PE = 32 * NP / kThreads;
#pragma unroll
  for (int e = 0; e < PE; ++e) {
    const int idx = threadIdx.x + e * kThreads;
    int i, k;
    if (!cols) {
      i = idx / NP;
      k = idx - i * NP;
    } else {
      k = idx >> 5;
      i = idx & 31;
    }
    P[i * (NP + 1) + k] = (i0 + i < n && k < n) ? v[e] : T(0);
  }
}

template <typename T, int NB, int NF, bool BF = false>
__global__ __launch_bounds__(kThreads) void k_schur_small(T* __restrict__ L, T* __restrict__ E,
                                                         const uint8_t* __restrict__ mask, int N, int n_, int nE, int s,
                                                         int off, int next_off, int nT, int first,
                                                         const T* __restrict__ Lsrc) {
  const int n = NF ? NF : n_;
  constexpr int NP = 32 * NB, PP = NP + 1;
  constexpr int PE = 32 * NP / kThreads;
  constexpr int NTRI = NB * (NB + 1) / 2;
  const int b = blockIdx.y;
  if (masked_out(mask, b)) return;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T* Pn = reinterpret_cast<T*>(smem_raw);  // four panels of 32 x PP
  const size_t nn = (size_t)n * n;
  T* Eb = E + (size_t)b * nE * nn;
  int task = first + blockIdx.x;
  const T* M[4];
  bool cols[4];
  int i0[4];
  int np;
  T* C;
  int tr, tc;
  bool diag;
  const bool target = task < nT * NTRI;
  if (target) {
    // L_j -= R R^T + Lc^T Lc  (R = block (j, j-s), Lc = block (j+s, j))
    const int u = task / NTRI;
    int q = task - u * NTRI;
    tr = 0;
    while (q > tr) { q -= tr + 1; ++tr; }
    tc = q;
    const int j = 2 * s * (u + 1) - 1;
    C = L + ((size_t)b * N + j) * nn;
    const T* R = Eb + (size_t)(off + (j - s) / s) * nn;
    const bool hasC = j + s < N;
    const T* Lc = hasC ? Eb + (size_t)(off + j / s) * nn : R;
    M[0] = R;  M[1] = R;  M[2] = Lc;  M[3] = Lc;
    cols[0] = false; cols[1] = false; cols[2] = true; cols[3] = true;
    i0[0] = 32 * tr; i0[1] = 32 * tc; i0[2] = 32 * tr; i0[3] = 32 * tc;
    np = hasC ? 2 : 1;
    diag = tr == tc;
  } else {
    // fill-in F -= R Lc  (node i: R = block (i+s, i), Lc = block (i, i-s))
    task -= nT * NTRI;
    const int f = task / (NB * NB);
    const int q = task - f * NB * NB;
    tr = q / NB;
    tc = q - tr * NB;
    const int i = s - 1 + 2 * s * (f + 1);
    const T* R = Eb + (size_t)(off + i / s) * nn;
    const T* Lc = Eb + (size_t)(off + (i - s) / s) * nn;
    C = Eb + (size_t)(next_off + (i - s) / (2 * s)) * nn;
    M[0] = R;  M[1] = Lc;  M[2] = R;  M[3] = Lc;
    cols[0] = false; cols[1] = true; cols[2] = false; cols[3] = true;
    i0[0] = 32 * tr; i0[1] = 32 * tc; i0[2] = 32 * tr; i0[3] = 32 * tc;
    np = 1;
    diag = false;
  }
  const int l = lane_id(), wave = wave_id();
  const int wi = wave >> 1, wj = wave & 1;
  // every load of the task at once: the panels, then this wave's C values.
  // (Diagonal tiles: panels 1 and 3 equal panels 0 and 2 and are neither
  // loaded nor stored.)
  T v[4][PE];
#pragma unroll
  for (int p = 0; p < 4; ++p)
    if (p < 2 * np && !(diag && (p & 1))) panel_load<T, NB>(v[p], M[p], cols[p], i0[p], n);
  // C values: the target's (the fill-in block receives its only update here,
  // F = -R Lc, so its entry contents are not read)
  T cv[4] = {T(0), T(0), T(0), T(0)};
  if (target) {
    // (out-of-place: the target is read from Lsrc, same layout)
    const T* Cin = (Lsrc != nullptr) ? Lsrc + (C - L) : C;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int rr = 32 * tr + 16 * wi + Mfma<T>::row(l, r), cc = 32 * tc + 16 * wj + Mfma<T>::col(l, r);
      cv[r] = Cin[min(rr, n - 1) * n + min(cc, n - 1)];
    }
  }
#pragma unroll
  for (int p = 0; p < 4; ++p)
#pragma unroll
    for (int e = 0; e < PE; ++e) pin_reg(v[p][e]);
#pragma unroll
  for (int r = 0; r < 4; ++r) pin_reg(cv[r]);
#pragma unroll
  for (int p = 0; p < 4; ++p)
    if (p < 2 * np && !(diag && (p & 1))) panel_store<T, NB>(Pn + p * 32 * PP, v[p], cols[p], i0[p], n);
  __syncthreads();
  typename Mfma<T>::acc_t acc = acc_zero<T>();
  for (int p = 0; p < np; ++p)
    schur_gemm16<T, BF>(acc, Pn + (2 * p) * 32 * PP + 16 * wi * PP, PP, 1,
                        Pn + (diag ? 2 * p : 2 * p + 1) * 32 * PP + 16 * wj * PP, 1, PP, NP);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int rr = 32 * tr + 16 * wi + Mfma<T>::row(l, r), cc = 32 * tc + 16 * wj + Mfma<T>::col(l, r);
    if (rr < n && cc < n && (!diag || cc <= rr)) C[rr * n + cc] = cv[r] - acc[r];
  }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
template <int NB>
static hipError_t set_schur_small_attrs() {
  const int lds = (int)schur_small_lds<float, NB>();
  hipError_t e = hipFuncSetAttribute((const void*)k_schur_small<float, NB, 0, true>,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e == hipSuccess)
    e = hipFuncSetAttribute((const void*)k_schur_small<float, NB, 32 * NB, true>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  return e;
}

// Whether a level's Schur updates (nodes = targets + fill-ins over the batch) take
// k_schur_blk rather than 16x16 tiles (k_schur_tile, nd_large.hip), which read each
// operand once per tile: where a level streams many blocks and the 64x64 tiles are
// all inside the block.  n = 128, FP64, levels of 256, 128, 64 and 32 nodes: 99, 58,
// 33 us (and 22 in 32x32 tiles with all of K staged in LDS) to 116, 60, 32 and 18.
// (n > 128 takes 16x16 tiles always, factor_level_large: n = 200, 32 nodes, 76 us to 54.)
static bool use_schur_blk(int nodes, int n, int esize) {
  return (n + 15) / 16 % 4 == 0 && (double)nodes * n * n * esize > 16.0 * 1024 * 1024;
}

// Whether a level's FP32 or BF16 Schur products take k_schur_small.
// FP32: blocks of one 32x32 tile that are not one 16x16 tile.  k_schur_tile reads
// each operand twice per output row of tiles and a wavefront has a quarter or a half
// of a short sum.  FP32 factor with FP64 pivots, n = 32, 8, 100, 16 x 64, 256 x 61 and
// 1024 x 64 blocks: 46, 81, 106, 430, 1610 us to 44, 78, 92, 287, 972; n = 17: 45, 80, 95,
// 356, 1279 to 45, 80, 88, 266, 868; n = 16, where three of four quarters of the tile are
// padding, 37, 64, 68, 154, 459 to 38, 65, 70, 164, 495.
// BF16: its panel loads repeat each operand per output tile, which only costs where
// the level streams many blocks; it wins up to about 12 MiB of the level's blocks
// (N=512, 1024), and for n <= 32 at every level: k_schur_blk's 64x64 output tiles
// leave three of four quarters outside a 32x32 block.  SOCU_SCHUR_SMALL=<nodes>
// replaces this rule by a node count (0 disables the small kernel).
static bool use_schur_small(int nodes, int n, bool bf16) {
  static int env = -2;
  if (env == -2) {
    const char* e = getenv("SOCU_SCHUR_SMALL");
    env = e ? (atoi(e) < 0 ? 0 : atoi(e)) : -1;
  }
  if (!bf16) return n > 16 && n <= 32;
  if (env >= 0) return nodes <= env;
  if (n <= 32) return true;
  return (double)nodes * n * n * sizeof(float) <= 12.0 * 1024 * 1024;
}

hipError_t init_blocked_kernels() {
  hipError_t e;
  if ((e = set_schur_small_attrs<1>()) != hipSuccess) return e;
  if ((e = set_schur_small_attrs<2>()) != hipSuccess) return e;
  if ((e = set_schur_small_attrs<3>()) != hipSuccess) return e;
  if ((e = set_schur_small_attrs<4>()) != hipSuccess) return e;
  return hipSuccess;
}

template <typename T, int NB, int NF>
static hipError_t factor_level_nb(T* L, T* E, const uint8_t* mask, int B, int N, int n, int lidx, int prec,
                                  hipStream_t st, hipEvent_t after_potrf, hipEvent_t after_trsm,
                                  hipEvent_t before_trsm, const T* Lsrc, const T* Esrc) {
  const int nE = (int)off_diag_storage_len(N);
  const int Lv = recursive_iterations(N);
  const Level lv = level_info(N, lidx);
  if (lv.dim <= 0 || B <= 0) return hipSuccess;
  const bool bf16 = (prec & kPrecBf16Schur) != 0 && sizeof(T) == 4;
  hipError_t ep = potrf_level<T>(L, mask, B, N, n, lidx, (prec & kPrecF64Pivots) != 0 && sizeof(T) == 4, Lsrc, 0, n, st);
  if (ep != hipSuccess) return ep;
  if (after_potrf != nullptr) {
    const hipError_t e = hipEventRecord(after_potrf, st);
    if (e != hipSuccess) return e;
  }
  if (lidx == Lv - 1) return hipGetLastError();
  if (before_trsm != nullptr) {
    const hipError_t e = hipStreamWaitEvent(st, before_trsm, 0);
    if (e != hipSuccess) return e;
  }
  ep = trsm_level<T>(L, E, Esrc, mask, B, N, n, lidx, st);
  if (ep != hipSuccess) return ep;
  if (after_trsm != nullptr) {
    const hipError_t e = hipEventRecord(after_trsm, st);
    if (e != hipSuccess) return e;
  }
  const int ntile = (n + kSTile - 1) / kSTile;
  const int ntri = ntile * (ntile + 1) / 2;
  const int nT = N / (2 * lv.s);
  int nF = 0;  // fill-in tasks
  for (int t = 1; t < lv.dim; ++t)
    if (lv.s - 1 + 2 * lv.s * t + lv.s < N) ++nF;
  const int tasks = nT * ntri + nF * ntile * ntile;
  if (tasks > 0) {
    kt_begin(kKcSchur, st);
    const int nodes = B * (nT + nF);
    const dim3 grid_blk(8 * schur_blk_per_xcd(nT, nF, ntile), B);
    // (pieces: as in schur_tiles)
    auto small = [&](auto bf) {
      const int count = nT * (NB * (NB + 1) / 2) + nF * NB * NB;
      for (int first = 0; first < count; first += kMaxGridTasks)
        hipLaunchKernelGGL((k_schur_small<T, NB, NF, decltype(bf)::value>), dim3(std::min(count - first, kMaxGridTasks), B),
                           dim3(kThreads), (schur_small_lds<T, NB>()), st, L, E, mask, N, n, nE, lv.s, lv.off, lv.next_off,
                           nT, first, Lsrc);
    };
    bool done = false;
    if constexpr (sizeof(T) == 4) {
      if (use_schur_small(nodes, n, bf16)) {
        if (bf16) small(std::true_type{});
        else if constexpr (NB == 1) small(std::false_type{});
        done = true;
      }
    }
    if (!bf16 && !done) {
      bool blk = false;
      if constexpr (NB % 2 == 0) blk = use_schur_blk(nodes, n, (int)sizeof(T));
      if (!blk) {
        ep = schur_tiles<T>(L, Lsrc, E, mask, B, N, n, lidx, nT, nF, st);
        if (ep != hipSuccess) return ep;
      } else if constexpr (NB % 2 == 0) {
        hipLaunchKernelGGL((k_schur_blk<T, NF, false>), grid_blk, dim3(kThreads), 0, st, L, E, mask, N, n, nE, lv.s,
                           lv.off, lv.next_off, nT, nF, ntile, Lsrc);
      }
    }
    if constexpr (sizeof(T) == 4) {
      if (bf16 && !done)
        hipLaunchKernelGGL((k_schur_blk<T, NF, true>), grid_blk, dim3(kThreads), 0, st, L, E, mask, N, n, nE, lv.s,
                           lv.off, lv.next_off, nT, nF, ntile, Lsrc);
    }
    kt_end(kKcSchur, st);
  }
  return hipGetLastError();
}

// One factor level for kMaxN < n <= kMaxNLarge: the diagonal blocks, R and Lc by
// nd_large.hip, then the Schur updates by 16x16 tiles.
template <typename T>
static hipError_t factor_level_large(T* L, T* E, const uint8_t* mask, int B, int N, int n, int lidx, hipStream_t st,
                                     hipEvent_t after_potrf, hipEvent_t after_trsm, hipEvent_t before_trsm) {
  const int Lv = recursive_iterations(N);
  const Level lv = level_info(N, lidx);
  if (lv.dim <= 0 || B <= 0) return hipSuccess;
  hipError_t e = before_trsm != nullptr ? hipStreamWaitEvent(st, before_trsm, 0) : hipSuccess;
  if (e == hipSuccess) e = factor_large<T>(L, E, mask, B, N, n, lidx, st);
  if (e == hipSuccess && after_potrf != nullptr) e = hipEventRecord(after_potrf, st);
  if (e == hipSuccess && after_trsm != nullptr) e = hipEventRecord(after_trsm, st);
  if (e != hipSuccess || lidx == Lv - 1) return e;
  const int nT = N / (2 * lv.s);
  int nF = 0;
  for (int t = 1; t < lv.dim; ++t)
    if (lv.s - 1 + 2 * lv.s * t + lv.s < N) ++nF;
  kt_begin(kKcSchur, st);
  e = schur_tiles<T>(L, nullptr, E, mask, B, N, n, lidx, nT, nF, st);
  kt_end(kKcSchur, st);
  return e;
}

template <typename T>
hipError_t factor_level_blocked(T* L, T* E, const uint8_t* mask, int B, int N, int n, int lidx, int prec,
                                hipStream_t st, hipEvent_t after_potrf, hipEvent_t after_trsm,
                                hipEvent_t before_trsm, const T* Lsrc, const T* Esrc) {
  if (n > kMaxN) {
    if (Lsrc != nullptr || Esrc != nullptr) return hipErrorInvalidValue;  // in place only
    return factor_level_large<T>(L, E, mask, B, N, n, lidx, st, after_potrf, after_trsm, before_trsm);
  }
  // small blocks in the storage precision (in place): one launch per level,
  // which applies the previous level's updates itself.  FP32 storage with FP64
  // pivots or BF16 Schur products takes the separate kernels.
  const bool separate = sizeof(T) == 4 && (prec & (kPrecF64Pivots | kPrecBf16Schur)) != 0;
  if (n <= kSmallUpN && !separate) {
    if (Lsrc != nullptr || Esrc != nullptr) return hipErrorInvalidValue;
    hipError_t e = before_trsm != nullptr ? hipStreamWaitEvent(st, before_trsm, 0) : hipSuccess;
    if (e == hipSuccess) e = small_up_level<T>(L, E, nullptr, mask, B, N, n, 0, lidx, st, nullptr, nullptr);
    if (e == hipSuccess && after_potrf != nullptr) e = hipEventRecord(after_potrf, st);
    if (e == hipSuccess && after_trsm != nullptr) e = hipEventRecord(after_trsm, st);
    return e;
  }
  // (FP64 blocks of n <= 64 have returned above)
  auto level = [&](auto nb, auto nf) {
    return factor_level_nb<T, decltype(nb)::value, decltype(nf)::value>(L, E, mask, B, N, n, lidx, prec, st, after_potrf,
                                                                        after_trsm, before_trsm, Lsrc, Esrc);
  };
  using std::integral_constant;
  if constexpr (sizeof(T) == 4) {
    if (n == 32) return level(integral_constant<int, 1>{}, integral_constant<int, 32>{});
    if (n < 32) return level(integral_constant<int, 1>{}, integral_constant<int, 0>{});
    if (n == 64) return level(integral_constant<int, 2>{}, integral_constant<int, 64>{});
    if (n < 64) return level(integral_constant<int, 2>{}, integral_constant<int, 0>{});
  }
  if (n == 96) return level(integral_constant<int, 3>{}, integral_constant<int, 96>{});
  if (n == 128) return level(integral_constant<int, 4>{}, integral_constant<int, 128>{});
  if (n < 96) return level(integral_constant<int, 3>{}, integral_constant<int, 0>{});
  return level(integral_constant<int, 4>{}, integral_constant<int, 0>{});
}

template <typename T>
hipError_t trtri_blocked(const T* L, T* W, const uint8_t* mask, int B, int N, int n, hipStream_t st) {
  if (n > kMaxN) {
    kt_begin(kKcForward, st);
    const hipError_t e = trtri_large<T>(L, W, mask, B, N, n, st);
    kt_end(kKcForward, st);
    return e;
  }
  kt_begin(kKcForward, st);
  const hipError_t e = trtri_blocks<T>(L, W, mask, B, N, n, 0, n, st);
  kt_end(kKcForward, st);
  return e;
}

template <typename T>
static hipError_t forward_step_parts(const T* L, const T* E, T* x, const uint8_t* mask, int B, int N, int n, int m,
                              int step, hipStream_t st, bool a, bool u) {
  if (n > kMaxN) {
    hipError_t e = hipSuccess;
    kt_begin(kKcForward, st);
    if (u && step >= 0) e = update_large<T>(E, x, mask, B, N, n, m, step, false, st);
    if (e == hipSuccess && a) e = apply_large<T>(L, x, mask, B, N, n, m, step + 1, false, st);
    kt_end(kKcForward, st);
    return e;
  }
  if (n <= kSmallN) return small_forward_step<T>(L, E, x, mask, B, N, n, m, step, st, u, a);
  return wide_forward_step<T>(L, E, x, mask, B, N, n, m, step, st, u, a);
}

template <typename T>
hipError_t forward_step_blocked(const T* L, const T* E, T* x, const uint8_t* mask, int B, int N, int n, int m,
                                int step, hipStream_t st, bool apply_next) {
  return forward_step_parts<T>(L, E, x, mask, B, N, n, m, step, st, apply_next, true);
}

template <typename T>
hipError_t forward_update_blocked(const T* L, const T* E, T* x, const uint8_t* mask, int B, int N, int n, int m,
                                  int step, hipStream_t st) {
  return forward_step_parts<T>(L, E, x, mask, B, N, n, m, step, st, false, true);
}

template <typename T>
hipError_t forward_apply_blocked(const T* L, const T* E, T* x, const uint8_t* mask, int B, int N, int n, int m,
                                 int level, hipStream_t st) {
  return forward_step_parts<T>(L, E, x, mask, B, N, n, m, level - 1, st, true, false);
}

template <typename T>
hipError_t backward_level_blocked(const T* L, const T* E, T* x, const uint8_t* mask, int B, int N, int n, int m,
                                  int lidx, hipStream_t st) {
  if (n > kMaxN) {
    const Level lv = level_info(N, lidx);
    hipError_t e = hipSuccess;
    kt_begin(kKcBackward, st);
    if (!(lv.dim == 1 && lv.s - 1 + lv.s >= N)) e = update_large<T>(E, x, mask, B, N, n, m, lidx, true, st);
    if (e == hipSuccess) e = apply_large<T>(L, x, mask, B, N, n, m, lidx, true, st);
    kt_end(kKcBackward, st);
    return e;
  }
  if (n <= kSmallN) return small_backward_level<T>(L, E, x, mask, B, N, n, m, lidx, st);
  return wide_backward_level<T>(L, E, x, mask, B, N, n, m, lidx, st);
}

hipError_t overlap_create(SweepOverlap& ov) {
  hipError_t e = hipStreamCreateWithFlags(&ov.side, hipStreamNonBlocking);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&ov.fork, hipEventDisableTiming);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&ov.join, hipEventDisableTiming);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&ov.ready, hipEventDisableTiming);
  for (int l = 0; l < kSweepMaxLevels && e == hipSuccess; ++l)
    e = hipEventCreateWithFlags(&ov.level[l], hipEventDisableTiming);
  if (e != hipSuccess) overlap_destroy(ov);
  return e;
}

void overlap_destroy(SweepOverlap& ov) {
  for (int l = 0; l < kSweepMaxLevels; ++l)
    if (ov.level[l]) (void)hipEventDestroy(ov.level[l]);
  if (ov.fork) (void)hipEventDestroy(ov.fork);
  if (ov.join) (void)hipEventDestroy(ov.join);
  if (ov.ready) (void)hipEventDestroy(ov.ready);
  if (ov.side) (void)hipStreamDestroy(ov.side);
  ov = SweepOverlap();
}

// The reference's fused factor_and_solve likewise interleaves the forward
// sweep into the factor's levels (block_tridiag_solver.py:926-1233).  Here
// the sweep runs on a second stream: the inverses of level l follow that
// level's potrf, its updates into the receiving blocks follow its trsm.
// Both read only finished factor blocks and write only x, which the factor
// does not touch.
template <typename T>
hipError_t factor_with_forward(T* L, T* E, T* x, const uint8_t* factor_mask, const uint8_t* sweep_mask, int B, int N,
                               int n, int m, int prec, const SweepOverlap& ov, hipStream_t st,
                               const std::function<hipError_t(hipStream_t)>* side_first, const T* Lsrc,
                               const T* Esrc) {
  const int Lv = recursive_iterations(N);
  hipError_t e = hipEventRecord(ov.fork, st);
  if (e == hipSuccess) e = hipStreamWaitEvent(ov.side, ov.fork, 0);
  if (e == hipSuccess && side_first != nullptr) e = (*side_first)(ov.side);
  if (e == hipSuccess && side_first != nullptr) e = hipEventRecord(ov.ready, ov.side);
  for (int l = 0; l < Lv && e == hipSuccess; ++l) {
    // one fork per level (each costs the main stream about 4 us in a graph):
    // behind level l's trsm the side stream applies level l and updates from it
    const bool last = l == Lv - 1;
    e = factor_level_blocked<T>(L, E, factor_mask, B, N, n, l, prec, st, last ? ov.level[l] : nullptr,
                                last ? nullptr : ov.level[l], (l == 0 && side_first != nullptr) ? ov.ready : nullptr,
                                l == 0 ? Lsrc : nullptr, l == 0 ? Esrc : nullptr);
    if (e == hipSuccess) e = hipStreamWaitEvent(ov.side, ov.level[l], 0);
    if (e == hipSuccess) e = forward_apply_blocked<T>(L, E, x, sweep_mask, B, N, n, m, l, ov.side);
    if (e == hipSuccess && !last) e = forward_update_blocked<T>(L, E, x, sweep_mask, B, N, n, m, l, ov.side);
  }
  if (e == hipSuccess) e = hipEventRecord(ov.join, ov.side);
  if (e == hipSuccess) e = hipStreamWaitEvent(st, ov.join, 0);
  return e;
}

template hipError_t factor_with_forward<float>(float*, float*, float*, const uint8_t*, const uint8_t*, int, int, int,
                                               int, int, const SweepOverlap&, hipStream_t,
                                               const std::function<hipError_t(hipStream_t)>*, const float*,
                                               const float*);
template hipError_t factor_with_forward<double>(double*, double*, double*, const uint8_t*, const uint8_t*, int, int,
                                                int, int, int, const SweepOverlap&, hipStream_t,
                                                const std::function<hipError_t(hipStream_t)>*, const double*,
                                                const double*);

template hipError_t trtri_blocked<float>(const float*, float*, const uint8_t*, int, int, int, hipStream_t);
template hipError_t trtri_blocked<double>(const double*, double*, const uint8_t*, int, int, int, hipStream_t);
template hipError_t factor_level_blocked<float>(float*, float*, const uint8_t*, int, int, int, int, int,
                                                hipStream_t, hipEvent_t, hipEvent_t, hipEvent_t, const float*,
                                                const float*);
template hipError_t factor_level_blocked<double>(double*, double*, const uint8_t*, int, int, int, int, int,
                                                 hipStream_t, hipEvent_t, hipEvent_t, hipEvent_t, const double*,
                                                 const double*);
template hipError_t forward_step_blocked<float>(const float*, const float*, float*, const uint8_t*, int, int, int, int,
                                                int, hipStream_t, bool);
template hipError_t forward_step_blocked<double>(const double*, const double*, double*, const uint8_t*, int, int, int,
                                                 int, int, hipStream_t, bool);
template hipError_t forward_update_blocked<float>(const float*, const float*, float*, const uint8_t*, int, int, int,
                                                  int, int, hipStream_t);
template hipError_t forward_update_blocked<double>(const double*, const double*, double*, const uint8_t*, int, int,
                                                   int, int, int, hipStream_t);
template hipError_t forward_apply_blocked<float>(const float*, const float*, float*, const uint8_t*, int, int, int,
                                                 int, int, hipStream_t);
template hipError_t forward_apply_blocked<double>(const double*, const double*, double*, const uint8_t*, int, int,
                                                  int, int, int, hipStream_t);
template hipError_t backward_level_blocked<float>(const float*, const float*, float*, const uint8_t*, int, int, int,
                                                  int, int, hipStream_t);
template hipError_t backward_level_blocked<double>(const double*, const double*, double*, const uint8_t*, int, int,
                                                   int, int, int, hipStream_t);

}  // namespace socu
