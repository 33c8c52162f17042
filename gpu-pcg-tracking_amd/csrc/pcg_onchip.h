// pcg_onchip.h -- block-row arithmetic shared by the on-chip PCG kernels
// (k_pcg_res.hip, k_pcg_team.hip) for gfx950.
//
// A knot b of the Schur system is served by a 16-lane group that matches a
// DPP row of the wave: lane i < 14 owns row i of block row b; lanes 14 and
// 15 carry zeros.  A vector (p, r, z, lambda) lives in registers, element i
// of knot b in lane i.  Each group serves 4 consecutive knots, so the
// neighbours of its inner knots are in its own registers and only the
// first and last knot's outer neighbours pass through LDS.  A 14x14 block
// times a vector is computed without
// moving the vector through LDS: under the DPP rotation row_ror:n lane i
// reads the lane src(i, n) = (i + n * d) mod 16 of its row (d = +-1, found
// once per kernel by rotating the lane id), so
//     (M x)_i = sum_{n=0..15} M(i, src(i, n)) * ror_n(x)_i
// with each lane holding its row of M "rotated": Mr[n] = M(i, src(i, n)),
// zero where src >= 14 or i >= 14.  One v_fmac_f32_dpp per term.
//
// Blocks of block row b, all in registers: D = S(b,b), P = Pinv(b,b) and
// L_b = S(b,b-1), rotated; the group also holds the L of the knot after its
// last.  S(b,b+1) = L_{b+1}^T is applied from the rows of L_{b+1} in
// "contribution" form: lane j forms L_{b+1}(j, i) x_j for the lane i that
// reads it under row_ror:n, i.e.
//     (L^T x)_i = sum_n ror_n(Lr[(16 - n) mod 16] * x)_i,
// so no transposed copy is held.  With four knots per group that is 208 of
// the 256 registers that two waves per SIMD have.
#pragma once
#include "common.h"

namespace mpc {
namespace onchip {

// direction of row_ror on this device: src(i, 1) - i (mod 16), 1 or 15.
// Must run with every lane of the row active; tid = the lane's thread index.
__device__ __forceinline__ uint32_t ror_step(uint32_t tid) {
  const int i = (int)(tid & 15u);
  const int s = __builtin_amdgcn_mov_dpp(i, 0x121, 0xF, 0xF, true);
  return (uint32_t)(s - i) & 15u;
}

// Two interleaved accumulations (independent dependency chains):
//   a += sum_{n=1..15} Ma[n] * ror_n(xa),  b += sum_{n=1..15} Mb[n] * ror_n(xb).
// A leading s_nop 4 covers the wait states required between a VALU (or
// EXEC) write and a DPP read of xa / xb.
__device__ __forceinline__ void rot_fma15x2(float &a, float xa, const float (&Ma)[16], float &b, float xb,
                                            const float (&Mb)[16]) {
#define MPC_RF2(n, oa, ob)                                                                        \
  "v_fmac_f32_dpp %0, %2, %" #oa " row_ror:" #n " row_mask:0xf bank_mask:0xf bound_ctrl:1\n" \
  "v_fmac_f32_dpp %1, %3, %" #ob " row_ror:" #n " row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
  asm("s_nop 4\n" MPC_RF2(1, 4, 11) MPC_RF2(2, 5, 12) MPC_RF2(3, 6, 13) MPC_RF2(4, 7, 14) MPC_RF2(5, 8, 15)
          MPC_RF2(6, 9, 16) MPC_RF2(7, 10, 17)
      : "+v"(a), "+v"(b)
      : "v"(xa), "v"(xb), "v"(Ma[1]), "v"(Ma[2]), "v"(Ma[3]), "v"(Ma[4]), "v"(Ma[5]), "v"(Ma[6]), "v"(Ma[7]),
        "v"(Mb[1]), "v"(Mb[2]), "v"(Mb[3]), "v"(Mb[4]), "v"(Mb[5]), "v"(Mb[6]), "v"(Mb[7]));
  asm("s_nop 4\n" MPC_RF2(8, 4, 12) MPC_RF2(9, 5, 13) MPC_RF2(10, 6, 14) MPC_RF2(11, 7, 15) MPC_RF2(12, 8, 16)
          MPC_RF2(13, 9, 17) MPC_RF2(14, 10, 18) MPC_RF2(15, 11, 19)
      : "+v"(a), "+v"(b)
      : "v"(xa), "v"(xb), "v"(Ma[8]), "v"(Ma[9]), "v"(Ma[10]), "v"(Ma[11]), "v"(Ma[12]), "v"(Ma[13]),
        "v"(Ma[14]), "v"(Ma[15]), "v"(Mb[8]), "v"(Mb[9]), "v"(Mb[10]), "v"(Mb[11]), "v"(Mb[12]), "v"(Mb[13]),
        "v"(Mb[14]), "v"(Mb[15]));
#undef MPC_RF2
}

// (Ma xa)_i and (Mb xb)_i for rotated rows Ma, Mb of full 16-lane rows
__device__ __forceinline__ void rot_mv2(const float (&Ma)[16], float xa, float &ya, const float (&Mb)[16], float xb,
                                        float &yb) {
  ya = Ma[0] * xa;
  yb = Mb[0] * xb;
  rot_fma15x2(ya, xa, Ma, yb, xb, Mb);
}

template <int CTRL>
__device__ __forceinline__ float dpp_f(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, false));
}

// total of the 16 lanes of each row, in every lane of the row (fixed order;
// each step adds two values in either order, so the lanes agree bitwise)
__device__ __forceinline__ float row_total(float v) {
  v += dpp_f<0xB1>(v);   // quad_perm [1,0,3,2]
  v += dpp_f<0x4E>(v);   // quad_perm [2,3,0,1]
  v += dpp_f<0x141>(v);  // row_half_mirror
  v += dpp_f<0x140>(v);  // row_mirror
  return v;
}

// wave64 sum, identical in every lane, in a fixed order: the rows, then
// (row0 + row1) + (row2 + row3)
__device__ __forceinline__ float wave_sum(float v) {
  v = row_total(v);
  const float r0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 0));
  const float r1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 16));
  const float r2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 32));
  const float r3 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 48));
  return (r0 + r1) + (r2 + r3);
}

// a condition that has the same value in every lane of the wave, in a scalar
// register (a branch on it leaves EXEC alone)
__device__ __forceinline__ bool uniform(bool v) { return __builtin_amdgcn_ballot_w64(v) != 0; }

// rotated rows of the column-major 14 x 14 block at base + off (floats);
// zeros where ok is false and for columns and lanes past 13
__device__ __forceinline__ void load_block(float (&R)[16], bool ok, uint32_t i, uint32_t d, const float *__restrict__ base,
                                           uint32_t off) {
#pragma unroll
  for (int n = 0; n < 16; ++n) R[n] = 0.f;
  if (ok) {
#pragma unroll
    for (int n = 0; n < 16; ++n) {
      const uint32_t j = (i + (uint32_t)n * d) & 15u;
      R[n] = base[off + i + (j < (uint32_t)NX ? NX * j : 0u)];
    }
#pragma unroll
    for (int n = 0; n < 16; ++n) R[n] = ((i + (uint32_t)n * d) & 15u) < (uint32_t)NX ? R[n] : 0.f;
  }
}

// Block rows of RK consecutive knots for lane i, and the L of the knot after
// them; zeros for absent ones and lanes >= 14.
template <int RK>
struct Rows {
  float D[RK][16], P[RK][16], L[RK + 1][16];

  // S, Pinv: of the instance; k0 the first knot, n its knots in all, own the
  // first knot past this workgroup's part
  __device__ __forceinline__ void load(const float *__restrict__ S, const float *__restrict__ Pinv, uint32_t k0,
                                       uint32_t own, uint32_t n, uint32_t i, uint32_t d) {
    const bool lane_ok = i < (uint32_t)NX;
#pragma unroll
    for (int t = 0; t < RK; ++t) {
      const uint32_t k = k0 + (uint32_t)t;
      const bool has = lane_ok && k < own;
      load_block(D[t], has, i, d, S, S_STRIDE * k + NXX);
      load_block(P[t], has, i, d, Pinv, S_STRIDE * k + NXX);
      load_block(L[t], has && k > 0, i, d, S, S_STRIDE * k);
    }
    const uint32_t k = k0 + RK;
    load_block(L[RK], lane_ok && k0 < own && k < n, i, d, S, S_STRIDE * k);
  }
};

// (D x + L xl) + M^T xr of one knot, M the rows of the next knot's left
// block: two direct chains, and the contributions of M's rows (header) in an
// even and an odd sum, m_0 + ror_2(m_2) of the even one a multiply-add; all
// four taken together step by step.  A pair of steps n, n + 1 (n odd): the products
// of the contributions come first, so that each DPP read is at least two
// instructions behind the write of what it reads.  (Of x and xl only the first
// statement makes sure itself; a copy of them that the compiler put right ahead
// of a later one would be found by tests/test_wait_states.py.)
#define MPC_DPPM " row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
#define MPC_PAIR(n, n1)                                                                                       \
  asm("v_mul_f32 %4, %13, %8\n"                                                                               \
      "v_mul_f32 %5, %14, %8\n"                                                                               \
      "v_fmac_f32_dpp %0, %6, %9 row_ror:" #n MPC_DPPM                                                        \
      "v_fmac_f32_dpp %1, %7, %11 row_ror:" #n MPC_DPPM                                                       \
      "v_add_f32_dpp %3, %4, %3 row_ror:" #n MPC_DPPM                                                         \
      "v_fmac_f32_dpp %0, %6, %10 row_ror:" #n1 MPC_DPPM                                                      \
      "v_fmac_f32_dpp %1, %7, %12 row_ror:" #n1 MPC_DPPM                                                      \
      "v_add_f32_dpp %2, %5, %2 row_ror:" #n1 MPC_DPPM                                                        \
      : "+v"(yd), "+v"(yl), "+v"(a), "+v"(b), "=&v"(t0), "=&v"(t1)                                            \
      : "v"(x), "v"(xl), "v"(xr), "v"(D[n]), "v"(D[n1]), "v"(L[n]), "v"(L[n1]), "v"(M[16 - n]), "v"(M[16 - n1]))
__device__ __forceinline__ float row_product(const float (&D)[16], float x, const float (&L)[16], float xl,
                                             const float (&M)[16], float xr) {
  float yd = D[0] * x, yl = L[0] * xl, a, b, t0 = M[15] * xr, t1 = M[14] * xr;
  asm("s_nop 1\n"
      "v_fmac_f32_dpp %0, %4, %8 row_ror:1" MPC_DPPM
      "v_fmac_f32_dpp %1, %5, %10 row_ror:1" MPC_DPPM
      "v_mov_b32_dpp %3, %6 row_ror:1" MPC_DPPM
      "v_mov_b32_dpp %2, %7 row_ror:2" MPC_DPPM
      "v_fmac_f32_dpp %0, %4, %9 row_ror:2" MPC_DPPM
      "v_fmac_f32_dpp %1, %5, %11 row_ror:2" MPC_DPPM
      "v_fmac_f32 %2, %12, %13\n"
      : "+v"(yd), "+v"(yl), "=&v"(a), "=&v"(b)
      : "v"(x), "v"(xl), "v"(t0), "v"(t1), "v"(D[1]), "v"(D[2]), "v"(L[1]), "v"(L[2]), "v"(M[0]), "v"(xr));
  MPC_PAIR(3, 4);
  MPC_PAIR(5, 6);
  MPC_PAIR(7, 8);
  MPC_PAIR(9, 10);
  MPC_PAIR(11, 12);
  MPC_PAIR(13, 14);
  asm("v_mul_f32 %3, %8, %9\n"
      "v_fmac_f32_dpp %0, %4, %6 row_ror:15" MPC_DPPM
      "v_fmac_f32_dpp %1, %5, %7 row_ror:15" MPC_DPPM
      "v_add_f32_dpp %2, %3, %2 row_ror:15" MPC_DPPM
      : "+v"(yd), "+v"(yl), "+v"(b), "=&v"(t0)
      : "v"(x), "v"(xl), "v"(D[15]), "v"(L[15]), "v"(M[1]), "v"(xr));
  return (yd + yl) + (a + b);
}
#undef MPC_PAIR
#undef MPC_DPPM

// z = P r
__device__ __forceinline__ float row_precond(const float (&P)[16], float r) {
  float z = P[0] * r;
#define MPC_RP(n, k) "v_fmac_f32_dpp %0, %1, %" #k " row_ror:" #n " row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
  asm("s_nop 1\n" MPC_RP(1, 2) MPC_RP(2, 3) MPC_RP(3, 4) MPC_RP(4, 5) MPC_RP(5, 6) MPC_RP(6, 7) MPC_RP(7, 8)
          MPC_RP(8, 9) MPC_RP(9, 10) MPC_RP(10, 11) MPC_RP(11, 12) MPC_RP(12, 13) MPC_RP(13, 14) MPC_RP(14, 15)
              MPC_RP(15, 16)
      : "+v"(z)
      : "v"(r), "v"(P[1]), "v"(P[2]), "v"(P[3]), "v"(P[4]), "v"(P[5]), "v"(P[6]), "v"(P[7]), "v"(P[8]), "v"(P[9]),
        "v"(P[10]), "v"(P[11]), "v"(P[12]), "v"(P[13]), "v"(P[14]), "v"(P[15]));
#undef MPC_RP
  return z;
}

// y = S x for the RK knots of a group; xm / xp the elements of the knots
// before and after them
template <int RK>
__device__ __forceinline__ void group_smv(const Rows<RK> &R, const float (&x)[RK], float xm, float xp,
                                          float (&y)[RK]) {
#pragma unroll
  for (int t = 0; t < RK; ++t)
    y[t] = row_product(R.D[t], x[t], R.L[t], t > 0 ? x[t - 1] : xm, R.L[t + 1], t < RK - 1 ? x[t + 1] : xp);
}

// z = Pinv r for the RK knots of a group
template <int RK>
__device__ __forceinline__ void group_precond(const Rows<RK> &R, const float (&r)[RK], float (&z)[RK]) {
#pragma unroll
  for (int t = 0; t < RK; ++t) z[t] = row_precond(R.P[t], r[t]);
}

}  // namespace onchip
}  // namespace mpc
