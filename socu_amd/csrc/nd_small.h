// What the kernels of the small-block paths share (nd_small.hip, n <= 32;
// nd_wide.hip, 32 < n <= 64): the systems of a launch, block accesses, and the
// panel factor with its rows in LDS.
#pragma once

#include <hip/hip_runtime.h>

#include "nd_common.h"
#include "nd_internal.h"
#include "nd_tile.h"

namespace socu {

// One system: the arrays of a task, Lin / Ein being where blocks are read
// that no earlier level has written (the sources of an out-of-place factor).
template <typename T>
struct SmallSys {
  T* L;
  const T* Lin;
  T* E;
  const T* Ein;
  T* x;
  int N, n, m;
};

// What a launch works on: B systems of one shape (probs NULL), or a table of
// uneven systems with a list of (system, task) pairs, one per workgroup.
template <typename T>
struct SmallArgs {
  T* L;
  const T* Lsrc;  // NULL: in place
  T* E;
  const T* Esrc;
  T* x;  // NULL: factor only
  const uint8_t* mask;
  int N, n, m, nE;
  const BatchProblem* probs;
  const int2* tasks;
  int solve;  // uneven systems: 0 ignores their x
};

// Element `off` of a block with a wave-uniform address (scalar base, 32-bit
// vector offset).
template <typename T>
__device__ __forceinline__ T ldg(const T* base, int off) {
  typedef const __attribute__((address_space(1))) char* gbytes;
  typedef const __attribute__((address_space(1))) T* gptr;
  return *(gptr)((gbytes)base + (unsigned)off * (unsigned)sizeof(T));
}
template <typename T>
__device__ __forceinline__ void stg(T* base, int off, T v) {
  typedef __attribute__((address_space(1))) char* gbytes;
  typedef __attribute__((address_space(1))) T* gptr;
  *(gptr)((gbytes)base + (unsigned)off * (unsigned)sizeof(T)) = v;
}
// Elements off, off + 1 of a block (no more than element alignment).
template <typename T>
struct Pair {
  typedef T type __attribute__((ext_vector_type(2)));
};
template <typename T>
__device__ __forceinline__ typename Pair<T>::type ldg2(const T* base, int off) {
  typedef typename Pair<T>::type v2 __attribute__((aligned(sizeof(T))));
  typedef const __attribute__((address_space(1))) char* gbytes;
  typedef const __attribute__((address_space(1))) v2* gptr;
  return *(gptr)((gbytes)base + (unsigned)off * (unsigned)sizeof(T));
}
// Element (row, col) of a block row of right-hand sides, m columns.  FAR: with a
// 64-bit offset, for block rows of 4 GiB and more (the sweeps take any m).
template <bool FAR, typename T>
__device__ __forceinline__ T ld_rhs(const T* y, int row, int m, int col) {
  typedef const __attribute__((address_space(1))) T* gptr;
  if constexpr (FAR) return ((gptr)y)[(unsigned long long)(unsigned)row * (unsigned)m + (unsigned)col];
  else return ldg(y, row * m + col);
}
template <bool FAR, typename T>
__device__ __forceinline__ void st_rhs(T* y, int row, int m, int col, T v) {
  typedef __attribute__((address_space(1))) T* gptr;
  if constexpr (FAR) ((gptr)y)[(unsigned long long)(unsigned)row * (unsigned)m + (unsigned)col] = v;
  else stg(y, row * m + col, v);
}
// Whether a launch needs it.
template <typename T>
bool far_rhs(int n, int m) {
  return (size_t)n * m * sizeof(T) > 0xffffffffu;
}
template <typename P>
__device__ __forceinline__ P* uniform_ptr(P* p) {
  const unsigned long long v = (unsigned long long)p;
  const unsigned lo = __builtin_amdgcn_readfirstlane((int)v), hi = __builtin_amdgcn_readfirstlane((int)(v >> 32));
  return (P*)(((unsigned long long)hi << 32) | lo);
}

template <typename T, int NP, int NC>
__device__ __forceinline__ void run_panel(T (&u)[16], T (&p)[NP][16], const T* urow, const T* prow) {
#pragma unroll
  for (int c = 0; c < NC; ++c) u[c] = urow[c];
#pragma unroll
  for (int c = 0; c < NC; ++c) p[0][c] = prow[c];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    pin_reg(u[c]);
    pin_reg(p[0][c]);
  }
  panel16<T, NP, NC>(u, p);
}

// Element offset of level l's segment of E, in blocks.
__device__ __forceinline__ int seg_offset(int N, int l) {
  int off = 0;
  for (int q = 0; q < l; ++q) off += (N >> q) - 1;
  return off;
}

// The system and task of this workgroup; false: nothing to do.
template <typename T>
__device__ __forceinline__ bool small_sys(const SmallArgs<T>& A, SmallSys<T>& Q, int& task) {
  if (A.probs != nullptr) {
    const int2 st = A.tasks[blockIdx.x];
    const int p = __builtin_amdgcn_readfirstlane(st.x);
    if (masked_out(A.mask, p)) return false;
    const BatchProblem P = A.probs[p];
    Q.L = uniform_ptr(static_cast<T*>(P.L));
    Q.E = uniform_ptr(static_cast<T*>(P.E));
    Q.x = A.solve ? uniform_ptr(static_cast<T*>(P.x)) : nullptr;
    Q.Lin = Q.L;
    Q.Ein = Q.E;
    Q.N = __builtin_amdgcn_readfirstlane(P.N);
    Q.n = __builtin_amdgcn_readfirstlane(P.n);
    Q.m = __builtin_amdgcn_readfirstlane(P.m);
    task = __builtin_amdgcn_readfirstlane(st.y);
    return true;
  }
  const int b = blockIdx.y;
  if (masked_out(A.mask, b)) return false;
  const size_t nn = (size_t)A.n * A.n, oL = (size_t)b * A.N * nn, oE = (size_t)b * A.nE * nn;
  Q.L = A.L + oL;
  Q.Lin = A.Lsrc != nullptr ? A.Lsrc + oL : Q.L;
  Q.E = A.E + oE;
  Q.Ein = A.Esrc != nullptr ? A.Esrc + oE : Q.E;
  Q.x = A.x != nullptr ? A.x + (size_t)b * A.N * A.n * A.m : nullptr;
  Q.N = A.N;
  Q.n = A.n;
  Q.m = A.m;
  task = blockIdx.x;
  return true;
}

// This wavefront's number, as a scalar.
__device__ __forceinline__ int wave_uniform() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

template <typename T>
SmallArgs<T> regular_args(T* L, T* E, T* x, const uint8_t* mask, int N, int n, int m, const T* Lsrc, const T* Esrc) {
  SmallArgs<T> A = {};
  A.L = L;
  A.Lsrc = Lsrc;
  A.E = E;
  A.Esrc = Esrc;
  A.x = x;
  A.mask = mask;
  A.N = N;
  A.n = n;
  A.m = x != nullptr ? m : 0;
  A.nE = (int)off_diag_storage_len(N);
  return A;
}

}  // namespace socu
