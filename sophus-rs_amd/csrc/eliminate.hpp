// Elimination of a few columns of a symmetric block by one wavefront, a row per lane: shared by
// the RCS factorization's diagonal blocks and the batched windows' dense factorization.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "block6.hpp"

namespace sgpu {

// f(integral_constant<int, I>) for I = B..E-1: indices that are constants, so that an array
// indexed by them stays in registers (a nest of this depth is past the loop unroller).
template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

// The value of lane N of each 16-lane row, in all its lanes.
template <int N>
__device__ __forceinline__ double row_value(double v) {
  constexpr int kNewBcast = 0x150 + N;  // DPP row_newbcast:N
  const int2 b = __builtin_bit_cast(int2, v);
  return __builtin_bit_cast(double,
                            make_int2(__builtin_amdgcn_mov_dpp(b.x, kNewBcast, 0xf, 0xf, true),
                                      __builtin_amdgcn_mov_dpp(b.y, kNewBcast, 0xf, 0xf, true)));
}

// acc += row_value<N>(v) * m in one instruction.  v must have been written two instructions
// before (the DPP read hazard); the callers' m depends on row_value of the same register.
template <int N>
__device__ __forceinline__ void fmac_row_value(double& acc, double v, double m) {
  asm("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
      : "+v"(acc)
      : "v"(v), "v"(m), "n"(N));
}

// Eliminates the first ncol (even) of kCols (<= 16) columns by one wavefront: lane i of each 16-lane
// row holds pivot row i in p (the same in every row of lanes), every lane one row below in q.
// No pivot test: a column is divided by what it finds.  The quotients are corrected by their
// remainders (4 more instructions a column).  Products with the reciprocal alone have the same
// errors (backward 5e-17 to 1e-16 at 24 to 180 rows and condition numbers 1e2 to 1e11, either way)
// and take 18.2 instead of 18.6 us in a round of panel steps, but whole calls the same (2000 cameras
// 1.000x, 500 cameras 0.998x); they would only move the results of long FP64 walks, where
// the last bits decide whether a step is taken.  On return p and q
// hold U = C L^-T and lane c (of each 16) the pivot d_c in dv.
//
// The next pivot's reciprocal is a chain of six dependent instructions; each is placed behind
// some of the column's independent updates (the scheduling barriers keep that order, which
// the compiler's scheduler would undo: it takes an asm statement's result as ready at once).
template <int kCols>
__device__ __forceinline__ void eliminate_columns(double (&p)[kCols], double (&q)[kCols], int ncol,
                                                  double& dv) {
  const int li = threadIdx.x & 15;
  double d = row_value<0>(p[0]), r = recip_nr(d);
  static_for<0, kCols / 2>([&](auto pair) __attribute__((always_inline)) {
    if (2 * pair >= ncol) return;
    static_for<2 * pair, 2 * pair + 2>([&](auto c) __attribute__((always_inline)) {
      dv = li == c ? d : dv;
      // -p / d and -q / d, each quotient corrected by its remainder
      double lp = -(p[c] * r), lq = -(q[c] * r);
      lp = fma(-fma(lp, d, p[c]), r, lp);
      lq = fma(-fma(lq, d, q[c]), r, lq);
      // update k of the column: p[c + 1], then p and q in turn
      constexpr int kUp = 2 * (kCols - 1 - c);
      auto update = [&](auto k) __attribute__((always_inline)) {
        constexpr int i = c + 1 + k / 2;
        if constexpr (k % 2 == 0) fmac_row_value<i>(p[i], p[c], lp);
        else fmac_row_value<i>(q[i], p[c], lq);
      };
      auto updates = [&](auto from, auto to) __attribute__((always_inline)) {
        static_for<(from < kUp ? int(from) : kUp), (to < kUp ? int(to) : kUp)>(update);
        __builtin_amdgcn_sched_barrier(0);
      };
      using std::integral_constant;
      if constexpr (kUp > 0) {
        updates(integral_constant<int, 0>{}, integral_constant<int, 4>{});
        d = row_value<(c + 1 < kCols ? c + 1 : 0)>(p[c + 1 < kCols ? c + 1 : 0]);
        updates(integral_constant<int, 4>{}, integral_constant<int, 6>{});
        r = __builtin_amdgcn_rcp(d);
        updates(integral_constant<int, 6>{}, integral_constant<int, 12>{});
        double e = fma(-d, r, 1.0);
        updates(integral_constant<int, 12>{}, integral_constant<int, 14>{});
        r = fma(r, e, r);
        updates(integral_constant<int, 14>{}, integral_constant<int, 16>{});
        e = fma(-d, r, 1.0);
        updates(integral_constant<int, 16>{}, integral_constant<int, 18>{});
        r = fma(r, e, r);
        updates(integral_constant<int, 18>{}, integral_constant<int, kUp>{});
      }
    });
  });
}

}  // namespace sgpu
