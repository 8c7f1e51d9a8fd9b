// Cholesky of a 16-column panel by one wavefront, without LDS traffic between
// its steps.
//
// CDNA's DPP row_newbcast gives every lane of a 16-lane DPP row the value of
// one lane of that row, as an operand modifier of the FP64 and FP32
// multiply-add itself.  With row r of a 16x16 diagonal tile in lane r of EACH
// of the wavefront's four DPP rows, the whole factor runs redundantly in all
// four and column k of L is always at hand: the update
//   u[q] -= L[r][k] L[q][k]
// is one v_fmac with lane q's L[.][k] broadcast.  The same broadcasts serve
// any further rows p ("payload", one per lane, 64 per register set):
//   p[k] *= 1/L[k][k],   p[q] -= p[k] L[q][k]   (q > k),   i.e.  p <- p L^-T.
// Payload rows are whatever needs L^-T from the right: panel rows below the
// diagonal tile (L_21 = A_21 L^-T), rows of the identity (giving U = L^-T, the
// transposed inverse), rows of R and of Lc^T.
//
// Why this form: one wavefront alone issues an independent FP64 multiply-add
// every 4.7 cycles (a dependent one every 8), a reciprocal square root with
// its correction takes 45, and a value that goes through LDS to the other
// lanes 112.  Publishing each column through LDS and reading it back entry by
// entry made a 32x32 factor with its inverse 13k cycles (400 per column);
// here a column costs its pivot chain (about 90 cycles), with the
// multiply-adds of the previous column underneath.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "nd_common.h"

namespace socu {

template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>)
template <int N, typename F>
__device__ __forceinline__ void static_for(F f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// acc -= (b of lane Q of this lane's DPP row) * c.  The two wait states a DPP
// read of b needs after a vector write of b are the caller's.  (The statements
// of a panel are volatile: their order is the schedule, see panel16.)
template <int Q>
__device__ __forceinline__ void fnma_row(double& acc, double b, double c) {
  asm volatile("v_fmac_f64_dpp %0, -%1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
               : "+v"(acc)
               : "v"(b), "v"(c), "n"(Q));
}
template <int Q>
__device__ __forceinline__ void fnma_row(float& acc, float b, float c) {
  asm volatile("v_fmac_f32_dpp %0, -%1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
               : "+v"(acc)
               : "v"(b), "v"(c), "n"(Q));
}
// v of lane Q of this lane's DPP row; NOPS wait states first.
template <int NOPS>
__device__ __forceinline__ void wait_states() {
  if constexpr (NOPS > 0) asm volatile("s_nop %0" ::"n"(NOPS > 0 ? NOPS - 1 : 0));
}
template <int Q>
__device__ __forceinline__ double bcast_row(double v) {
  double o;
  asm volatile("v_mov_b64_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf" : "=v"(o) : "v"(v), "n"(Q));
  return o;
}
template <int Q>
__device__ __forceinline__ float bcast_row(float v) {
  float o;
  asm volatile("v_mov_b32_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf" : "=v"(o) : "v"(v), "n"(Q));
  return o;
}

// 1/sqrt(x) (double: as rsqrt_t computes it), with fill(integral_constant i)
// between its dependent operations (i = 0 .. kFillSteps - 1).
constexpr int kFillSteps = 6;
#define SOCU_FILL(i)                             \
  __builtin_amdgcn_sched_barrier(0);             \
  fill(std::integral_constant<int, i>{});        \
  __builtin_amdgcn_sched_barrier(0)
template <typename Fill>
__device__ __forceinline__ double rsqrt_filled(double x, Fill fill) {
  const double y = __builtin_amdgcn_rsq(x);
  SOCU_FILL(0);
  const double t = -x * y;
  SOCU_FILL(1);
  const double e = fma(t, y, 1.0);
  SOCU_FILL(2);
  const double h = fma(e, 0.375, 0.5);
  SOCU_FILL(3);
  const double g = e * h;
  SOCU_FILL(4);
  const double r = fma(y, g, y);
  SOCU_FILL(5);
  return r;
}
// (float: one Newton step on the hardware's 1-ulp estimate; its operations
// find room between the multiply-adds)
template <typename Fill>
__device__ __forceinline__ float rsqrt_filled(float x, Fill fill) {
  const float y = __builtin_amdgcn_rsqf(x);
  SOCU_FILL(0);
  const float t = -x * y;
  SOCU_FILL(1);
  const float e = fmaf(t, y, 1.0f), h = 0.5f * y;
  SOCU_FILL(2);
  const float r = fmaf(h, e, y);
  SOCU_FILL(3);
  SOCU_FILL(4);
  SOCU_FILL(5);
  return r;
}
#undef SOCU_FILL

// How many of `total` independent multiply-adds go to each of the 9 places of
// a pivot step's chain: 0 before the pivot's broadcast (its operand needs two
// wait states), 1 behind it, 2 behind the hardware estimate, 3..7 behind the
// correction's operations, 8 behind the scaled column (two wait states
// again).  First what the latencies ask for, then the rest evenly.
constexpr int kPlaces = 9;
struct PanelPlan {
  int begin[kPlaces + 1];
};
constexpr PanelPlan panel_plan(int total) {
  const int want[kPlaces] = {2, 1, 3, 1, 1, 1, 1, 1, 2};
  const int order[kPlaces] = {0, 8, 2, 1, 3, 4, 5, 6, 7};
  int got[kPlaces] = {};
  int left = total;
  for (int o = 0; o < kPlaces; ++o) {
    const int w = want[order[o]] < left ? want[order[o]] : left;
    got[order[o]] = w;
    left -= w;
  }
  for (int i = 1; left > 0; i = i % (kPlaces - 1) + 1) {
    ++got[i];
    --left;
  }
  PanelPlan p = {};
  for (int i = 0; i < kPlaces; ++i) p.begin[i + 1] = p.begin[i] + got[i];
  return p;
}

// u: row (lane % 16) of the 16x16 tile, in every DPP row; on return its
// entries c <= lane % 16 hold that row of L (the others are not meaningful;
// what the tile's strict upper triangle holds on entry is not used either).
// p[j]: NP payload rows per lane, p[j] <- p[j] L^-T.
// NC: columns of the panel (a tile whose last 16 - NC rows and columns are
// identity padding needs no steps for them; entries from NC on are untouched).
// All 64 lanes must be active.
//
// Step k's multiply-adds other than the one that gives the next pivot are
// spread between the dependent operations of the next pivot's reciprocal
// square root (left to itself the compiler moves each one down to the first
// use of its result, and the chain then waits out every latency).
template <typename T, int NP, int NC = 16>
__device__ __forceinline__ void panel16(T (&u)[16], T (&p)[NP][16]) {
  wait_states<2>();
  T inv = rsqrt_filled(bcast_row<0>(u[0]), [](auto) {});
  T lk = u[0] * inv, pk[NP];
#pragma unroll
  for (int j = 0; j < NP; ++j) pk[j] = p[j][0] * inv;
  __builtin_amdgcn_sched_barrier(0);
  wait_states<2>();
  static_for<NC>([&](auto kc) {
    constexpr int k = decltype(kc)::value;
    u[k] = lk;  // row k itself: piv / sqrt(piv)
#pragma unroll
    for (int j = 0; j < NP; ++j) p[j][k] = pk[j];
    if constexpr (k + 1 < NC) {
      fnma_row<k + 1>(u[k + 1], lk, lk);
      // the updates left: payload entry k + 1 of each set (the next step
      // multiplies it), then u[k+2..], then the rest of the payload
      constexpr int nu = NC - 2 - k, total = NP + nu + NP * nu;
      constexpr PanelPlan plan = panel_plan(total);
      auto place = [&](auto pc) {
        constexpr int b = plan.begin[decltype(pc)::value], n = plan.begin[decltype(pc)::value + 1] - b;
        static_for<n>([&](auto ic) {
          constexpr int i = b + decltype(ic)::value;
          if constexpr (i < NP) {
            fnma_row<k + 1>(p[i][k + 1], lk, pk[i]);
          } else if constexpr (i < NP + nu) {
            constexpr int q = k + 2 + i - NP;
            fnma_row<q>(u[q], lk, lk);
          } else {
            constexpr int e = i - NP - nu, j = e / (nu > 0 ? nu : 1), q = k + 2 + e % (nu > 0 ? nu : 1);
            fnma_row<q>(p[j][q], lk, pk[j]);
          }
        });
      };
      place(std::integral_constant<int, 0>{});
      constexpr int n0 = plan.begin[1], n8 = plan.begin[9] - plan.begin[8];
      wait_states<(n0 < 2) ? 2 - n0 : 0>();
      const T piv = bcast_row<k + 1>(u[k + 1]);
      place(std::integral_constant<int, 1>{});
      __builtin_amdgcn_sched_barrier(0);
      inv = rsqrt_filled(piv, [&](auto ic) { place(std::integral_constant<int, 2 + decltype(ic)::value>{}); });
      const T nlk = u[k + 1] * inv;
      T npk[NP];
#pragma unroll
      for (int j = 0; j < NP; ++j) npk[j] = p[j][k + 1] * inv;
      __builtin_amdgcn_sched_barrier(0);
      place(std::integral_constant<int, 8>{});
      wait_states<(n8 + NP < 2) ? 2 - n8 - NP : 0>();
      lk = nlk;
#pragma unroll
      for (int j = 0; j < NP; ++j) pk[j] = npk[j];
    }
  });
}

}  // namespace socu
