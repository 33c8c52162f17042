// gj16.h -- 14x14 block algebra inside a 16-lane group (gfx950): lane j
// holds column j of a block in registers; a pivot column is broadcast to
// the group by DPP, in the multiply-adds themselves (Gauss-Jordan) or ahead of
// them (the whitening factor), so neither needs an LDS buffer or a barrier.  Used by
// the Schur formation (k_schur.hip), the split PCG (k_pcg_split.hip) and
// the direct block-tridiagonal solve (k_direct.hip).
#pragma once
#include "common.h"

namespace mpc {

// Value of lane P of the calling lane's 16-lane group by DPP row_newbcast:P
// (dpp_ctrl 0x150 + P, gfx90a and later): lane P of each 16-lane row to the
// whole row, one VALU instruction with no trip through the LDS pipeline.
// Lane P must be active.
template <int P>
__device__ __forceinline__ float bcast16_dpp(float v) {
  static_assert(P >= 0 && P < 16, "row lane");
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x150 + P, 0xf, 0xf, true));
}

// bcast16_dpp with the lane p given as a value that is a constant after loop
// unrolling (the instruction takes the lane as an immediate)
__device__ __forceinline__ float bcast_dyn16(float v, int p) {
#define MPC_BCASE(P) \
  case P: return bcast16_dpp<P>(v);
  switch (p) {
    MPC_BCASE(0) MPC_BCASE(1) MPC_BCASE(2) MPC_BCASE(3) MPC_BCASE(4) MPC_BCASE(5) MPC_BCASE(6) MPC_BCASE(7)
    MPC_BCASE(8) MPC_BCASE(9) MPC_BCASE(10) MPC_BCASE(11) MPC_BCASE(12) MPC_BCASE(13) MPC_BCASE(14)
    default: return bcast16_dpp<15>(v);
  }
#undef MPC_BCASE
}

// Materialise values at this point of the program: keeps the compiler from
// sinking their computation to a later (conditional) use, which would keep
// all of its inputs alive in registers.
template <int n>
__device__ __forceinline__ void pin(float (&v)[n]) {
#pragma unroll
  for (int r = 0; r < n; ++r) asm volatile("" : "+v"(v[r]));
}

// x -= c xp and a -= c ap for six rows (or one) of a pivot step, c the row's
// element of the pivot column: lane p's a, by DPP.  (The s_nop: a DPP read
// needs two wait states after the write of what it reads.)
#define MPC_GJ_ROW(k)                                                                                        \
  "v_fmac_f32_dpp %[x" #k "], %[a" #k "], -%[xp] row_newbcast:%c[p] row_mask:0xf bank_mask:0xf bound_ctrl:1\n" \
  "v_fmac_f32_dpp %[a" #k "], %[a" #k "], -%[ap] row_newbcast:%c[p] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
#define MPC_GJ_OPS(k) [x##k] "+v"(x[(r0 + k) % n]), [a##k] "+v"(a[(r0 + k) % n])
template <int n, int p, int r0>
__device__ __forceinline__ void gj_rows6(float (&x)[NX], float (&a)[NX], float xp, float ap) {
  asm("s_nop 1\n" MPC_GJ_ROW(0) MPC_GJ_ROW(1) MPC_GJ_ROW(2) MPC_GJ_ROW(3) MPC_GJ_ROW(4) MPC_GJ_ROW(5)
      : MPC_GJ_OPS(0), MPC_GJ_OPS(1), MPC_GJ_OPS(2), MPC_GJ_OPS(3), MPC_GJ_OPS(4), MPC_GJ_OPS(5)
      : [xp] "v"(xp), [ap] "v"(ap), [p] "i"(p));
}
template <int n, int p, int r0>
__device__ __forceinline__ void gj_rows1(float (&x)[NX], float (&a)[NX], float xp, float ap) {
  asm("s_nop 1\n" MPC_GJ_ROW(0) : MPC_GJ_OPS(0) : [xp] "v"(xp), [ap] "v"(ap), [p] "i"(p));
}
#undef MPC_GJ_OPS
#undef MPC_GJ_ROW

template <int n, int p>
__device__ __forceinline__ void gj_step(float (&a)[NX], float (&x)[NX]) {
  static_assert(n == NX || n == NU, "6 + 6 + 1 or 6 rows beside the pivot's");
  const float inv = 1.f / bcast_dyn16(a[p], p);
  const float ap = a[p] * inv, xp = x[p] * inv;
  // from the next pivot's row on, so that its division can start
  gj_rows6<n, p, p + 1>(x, a, xp, ap);
  if constexpr (n == NX) {
    gj_rows6<n, p, p + 7>(x, a, xp, ap);
    gj_rows1<n, p, p + 13>(x, a, xp, ap);
  }
  a[p] = ap;
  x[p] = xp;
}

template <int n, int p = 0>
__device__ __forceinline__ void gj_steps(float (&a)[NX], float (&x)[NX]) {
  if constexpr (p < n) {
    gj_step<n, p>(a, x);
    gj_steps<n, p + 1>(a, x);
  }
}

// Gauss-Jordan inverse of an n x n matrix (n <= 14) held by columns: lane
// j < n holds column j of M in a[0..n) (lanes >= n hold a copy of column
// n-1, which no lane reads); returns column j of M^-1 in x.  Every lane of
// the group must be active.
template <int n>
__device__ __forceinline__ void gj_inverse(int lane, float (&a)[NX], float (&x)[NX]) {
  const int j = lane < n ? lane : n - 1;
#pragma unroll
  for (int r = 0; r < n; ++r) x[r] = (r == j) ? 1.f : 0.f;
  gj_steps<n>(a, x);
}

// Whitening factor of a symmetric positive definite n x n matrix M (n <=
// 14) held by columns (lane j < n: column j in a; lanes >= n a copy of
// column n-1): Gauss elimination of [M | I] without pivoting, each pivot row
// scaled by the pivot's inverse square root once final.  Afterwards lane j
// holds row j of W = U^-1 in x, where M = U^T U (Cholesky, U upper
// triangular; the scaled rows of the left half are the rows of U), so
// W^T M W = I; a is destroyed.  Every lane of the group must be active.
// The pivot's reciprocal and inverse square root are the hardware's
// (v_rcp_f32, v_rsq_f32: 1 ulp), not the correctly rounded sequences: W is
// this build's own factor (no reference operation), and a one-ulp change
// of a multiplier is a rounding-level change of M.
template <int n>
__device__ __forceinline__ void chol_inv_rows(int lane, float (&a)[NX], float (&x)[NX]) {
  const int j = lane < n ? lane : n - 1;
#pragma unroll
  for (int r = 0; r < NX; ++r) x[r] = (r == j) ? 1.f : 0.f;
#pragma unroll
  for (int p = 0; p < n; ++p) {
    float pc[NX];
#pragma unroll
    for (int r = p; r < n; ++r) pc[r] = bcast_dyn16(a[r], p);
    const float inv = __builtin_amdgcn_rcpf(pc[p]);
    const float s = __builtin_amdgcn_rsqf(pc[p]);
    const float ap = a[p], xp = x[p];
#pragma unroll
    for (int r = p + 1; r < n; ++r) {
      const float m = pc[r] * inv;
      a[r] -= m * ap;
      x[r] -= m * xp;
    }
    a[p] = ap * s;
    x[p] = xp * s;
    pin(a);
    pin(x);
  }
}

}  // namespace mpc
