// k_direct.hip -- direct solve of the Schur system S lambda = gamma of every
// instance by block LDL^T (block Thomas) of the symmetric positive definite
// A = -S (gfx950).
//
// Factorisation (A_b = -S(b,b), B_b = -S(b,b-1)):
//   D_0 = A_0,   E_b = B_b D_{b-1}^-1,   D_b = A_b - E_b B_b^T,
// with D_b^-1 by Gauss-Jordan in registers (D_b is SPD: no pivoting); E_b
// and D_b^-1 are stored in the workspace (the S layout: E_b in the left
// block slot, D_b^-1 in the diagonal slot, a vector in the right slot).
// Solve of A x = r:
//   forward   y_b = r_b - E_b y_{b-1},   z_b = D_b^-1 y_b
//   backward  x_{N-1} = z_{N-1},   x_b = z_b - E_{b+1}^T x_{b+1}
// (from the other end E_b couples b to b + 1 in the same way, with B_{b+1}^T,
// and is kept in row b + 1), with r = -gamma, then `refine` steps of iterative refinement: the
// residual -gamma + S lambda in fp64 from the fp32 blocks, the same solve on
// it, lambda += x.  The fp32 elimination alone is off by about cond(S) x eps
// (1e-4..1e-2 relative on these systems); each step multiplies the error by
// about that factor, down to the fp32 storage of lambda.
//
// Mapping: one wave per instance, or (direct_both_ends) two, one from each end,
// which meet in the middle knot (a block tridiagonal system eliminates from both
// ends with the same operations, so the chain is half as long); instances longest first (few waves, one per SIMD: the sweeps are
// bound by their dependent chains, so what counts is the instructions and
// latencies of a step, below).  The residual is formed for
// all knots of all instances at once, one group per knot.
//
// Reference: the QDLDL path of sqpSolve (PCG_SOLVE = 0, toplevel.cuh:160-215,
// :314-335) solves the same system by a sparse LDL^T on the host.
#include <utility>

#include "common.h"
#include "gj16.h"

namespace mpc {

namespace {

constexpr int GROUP = 16;
constexpr int GROUPS_PER_WG = 4;
constexpr int WG = GROUP * GROUPS_PER_WG;

__device__ __forceinline__ float *slot_z(float *work, size_t row) { return work + (size_t)S_STRIDE * row + 2 * NXX; }

// the instance of a wave
struct Pick {
  uint32_t inst, K0, N;
  bool live;
};

__device__ __forceinline__ Pick pick_instance(const Batch &b, const uint32_t *order, const uint32_t *status,
                                              uint32_t slot) {
  Pick p;
  p.inst = order ? order[slot] : slot;
  p.K0 = inst_first(b, p.inst);
  p.N = inst_len(b, p.inst);
  p.live = !(status && !(status[p.inst] & ST_ACTIVE));
  return p;
}

// One side's elimination: chain positions 0 .. n are the knots from its end of
// the instance to the meeting knot (n), side 1 counting backwards.  With one
// side that is the last knot, and nothing meets there.
struct Chain {
  uint32_t side, n, N;
  // the knot at position k
  __device__ __forceinline__ uint32_t knot(uint32_t k) const { return side ? N - 1u - k : k; }
  // the block row that holds the coupling of positions k - 1 and k (and, in
  // the workspace, E of position k); row 0, with zeros, for k = 0
  __device__ __forceinline__ uint32_t link(uint32_t k) const { return k == 0 ? 0u : side ? N - k : k; }
};

template <bool TWO>
__device__ __forceinline__ Chain chain_of(uint32_t N, uint32_t side) {
  const uint32_t m = TWO ? N / 2u : N - 1u;  // the meeting knot
  return Chain{side, side ? N - 1u - m : m, N};
}

// ---- factorisation -----------------------------------------------------------
// Lane 16 q + j (q = 0..3) holds, for column j of a block, the rows
// r = 4 t + q (t = 0..3, r < 14): the products and the Gauss-Jordan updates
// of a column are split over four lanes, one row of 16 lanes per quarter.
// Per knot:
//   E_b = B_b D_{b-1}^-1: the lane's rows of B_b and its column of D_{b-1}^-1
//     from LDS (the latter written by the quarters after their inverse);
//   D_b = A_b - E_b B_b^T: the element E(r, m) is in lane m of the lane's own
//     row, so the 14 x 4 multiply-adds take it by DPP row_newbcast:m;
//   D_b^-1 by Gauss-Jordan, 14 pivots.  In step P the updates of the lane's
//     rows take column P by DPP (in the multiply-add itself), and row P comes
//     from its quarter by ds_bpermute (about 64 clocks).  Row P + 1 is updated
//     first and sent; its pivot is read by readlane and inverted between the
//     updates of the other rows, which cover both latencies.
// Every element sees the operations of a one-lane-per-column elimination in
// their order (a product m by m from zero, a pivot after the other).
// N = 512: 3.4 -> 1.27 us per knot (before: pivot columns by ds_swizzle, a
// division on the chain, 528 clocks per pivot).
constexpr int RS = 16;  // LDS row stride of a block (16-byte aligned rows)
struct alignas(16) FacWaveLds {
  float B[2][NX * RS + RS];  // B by rows: B(r, c) at c + RS r, knots alternating (the last RS: unused lanes' writes)
  float Dinv[NX * RS];       // the D^-1 before by columns: (m, j) at m + RS j
};
template <bool TWO>
struct alignas(16) DirectLds {
  FacWaveLds side[TWO ? 2 : 1];
  float meet[4][64];  // side 1's part of D at the meeting knot, by slot and lane
  float v[16], x[16]; // in the sweeps: its part of y there; y, then x
};

__device__ __forceinline__ float lane_value(float v, uint32_t byte_addr) {
  return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((int)byte_addr, __builtin_bit_cast(int, v)));
}
template <int l>
__device__ __forceinline__ float read_lane(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}

// a pivot whose inverse pivot_rest gives as the division does (below)
__device__ __forceinline__ bool mid_range(float v) {
  return ((__builtin_bit_cast(uint32_t, v) >> 23) & 255u) - 80u < 95u;  // 2^-47 <= |v| < 2^48
}

#define MPC_NB " row_newbcast:%c[l] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
// One slot of a pivot step: x -= column * xp, a -= column * ap, the column's
// element by DPP from lane l of the row; then the next pivot from lane pl of
// a.  A DPP read needs two wait states after the write of what it reads.  From
// step 1 on they are there: a was written in the step before, at least the two
// products ap and xp ago.  In step 0 the compiler's copies and negations of
// the block may stand right before the asm (it does not see the read inside),
// so it begins with an s_nop, as does pivot_rest's.  Reading the pivot takes two
// wait states after the v_readlane: pivot_rest has three instructions ahead of
// it, but DIV divides by it at once.  (tests/test_wait_states.py checks the
// listing.)
#define MPC_PIVOT_FIRST(before, behind)           \
  asm(before                                      \
      "v_fmac_f32_dpp %[x], %[a], -%[xp]" MPC_NB  \
      "v_fmac_f32_dpp %[a], %[a], -%[ap]" MPC_NB  \
      "s_nop 0\n"                                 \
      "v_readlane_b32 %[p], %[a], %[pl]\n"        \
      behind                                      \
      : [x] "+v"(x), [a] "+v"(a), [p] "=s"(piv)   \
      : [xp] "v"(xp), [ap] "v"(ap), [l] "i"(l), [pl] "i"(pl))
template <bool DIV, int l, int pl>
__device__ __forceinline__ float pivot_first(float &x, float &a, float xp, float ap) {
  float piv;
  if constexpr (DIV)
    MPC_PIVOT_FIRST("s_nop 1\n", "s_nop 1\n");
  else if constexpr (l == 0)
    MPC_PIVOT_FIRST("s_nop 1\n", "");
  else
    MPC_PIVOT_FIRST("", "");
  return piv;
}
#undef MPC_PIVOT_FIRST

// The other three slots of the step, with the next pivot's inverse between
// them: v_rcp_f32, one refinement and two residual steps, which is the
// division's own sequence without its scaling and fix-up, so the correctly
// rounded 1 / piv for a mid_range pivot.  Last, row P (quarter mask) becomes
// [ap, xp] in its slot.  In a step that is not the last of its slot, that is
// the slot of row P + 1 (pivot_first's), else one of the three.
#define MPC_SLOT_X(k) "v_fmac_f32_dpp %[x" #k "], %[a" #k "], -%[xp]" MPC_NB
#define MPC_SLOT_A(k) "v_fmac_f32_dpp %[a" #k "], %[a" #k "], -%[ap]" MPC_NB
#define MPC_PIVOT_REST                          \
  MPC_SLOT_X(0) MPC_SLOT_X(1) MPC_SLOT_X(2)     \
  "v_rcp_f32 %[r], %[p]\n"                      \
  MPC_SLOT_A(0)                                 \
  "v_fma_f32 %[t], -%[p], %[r], 1.0\n"          \
  MPC_SLOT_A(1)                                 \
  "v_fma_f32 %[r], %[t], %[r], %[r]\n"          \
  MPC_SLOT_A(2)                                 \
  "v_fma_f32 %[t], -%[p], %[r], 1.0\n"          \
  "v_fma_f32 %[i], %[t], %[r], %[r]\n"          \
  "v_fma_f32 %[t], -%[p], %[i], 1.0\n"          \
  "v_fma_f32 %[i], %[t], %[r], %[i]\n"
#define MPC_PIVOT_REST_OTHER(before)                                                                                \
  asm(before MPC_PIVOT_REST                                                                                         \
      "v_cndmask_b32_e64 %[ac], %[ac], %[ap], %[m]\n"                                                               \
      "v_cndmask_b32_e64 %[xc], %[xc], %[xp], %[m]\n"                                                               \
      : [x0] "+v"(x0), [a0] "+v"(a0), [x1] "+v"(x1), [a1] "+v"(a1), [x2] "+v"(x2), [a2] "+v"(a2), [xc] "+v"(xc),     \
        [ac] "+v"(ac), [i] "=&v"(inv), [r] "=&v"(r), [t] "=&v"(t)                                                   \
      : [xp] "v"(xp), [ap] "v"(ap), [p] "s"(piv), [m] "s"(mask), [l] "i"(l))
template <int l>
__device__ __forceinline__ float pivot_rest(float &x0, float &a0, float &x1, float &a1, float &x2, float &a2, float xp,
                                            float ap, float piv, float &xc, float &ac, uint64_t mask) {
  float inv, r, t;
  if constexpr (l == 0)
    MPC_PIVOT_REST_OTHER("s_nop 1\n");
  else
    MPC_PIVOT_REST_OTHER("");
  return inv;
}
#undef MPC_PIVOT_REST_OTHER
// row P in the first of the three slots (not in step 0, whose row 0 and row 1
// are in one slot)
template <int l>
__device__ __forceinline__ float pivot_rest(float &x0, float &a0, float &x1, float &a1, float &x2, float &a2, float xp,
                                            float ap, float piv, uint64_t mask) {
  static_assert(l > 0, "no wait states ahead of the first DPP read");
  float inv, r, t;
  asm(MPC_PIVOT_REST
      "v_cndmask_b32_e64 %[a0], %[a0], %[ap], %[m]\n"
      "v_cndmask_b32_e64 %[x0], %[x0], %[xp], %[m]\n"
      : [x0] "+v"(x0), [a0] "+v"(a0), [x1] "+v"(x1), [a1] "+v"(a1), [x2] "+v"(x2), [a2] "+v"(a2), [i] "=&v"(inv),
        [r] "=&v"(r), [t] "=&v"(t)
      : [xp] "v"(xp), [ap] "v"(ap), [p] "s"(piv), [m] "s"(mask), [l] "i"(l));
  return inv;
}
#undef MPC_PIVOT_REST
#undef MPC_SLOT_A
#undef MPC_SLOT_X
// x -= column * xp (the last pivot: A is not used after it)
template <int l>
__device__ __forceinline__ void pivot_last(float (&x)[4], const float (&a)[4], float xp) {
  asm("s_nop 1\n"
      "v_fmac_f32_dpp %[x0], %[a0], -%[xp]" MPC_NB
      "v_fmac_f32_dpp %[x1], %[a1], -%[xp]" MPC_NB
      "v_fmac_f32_dpp %[x2], %[a2], -%[xp]" MPC_NB
      "v_fmac_f32_dpp %[x3], %[a3], -%[xp]" MPC_NB
      : [x0] "+v"(x[0]), [x1] "+v"(x[1]), [x2] "+v"(x[2]), [x3] "+v"(x[3])
      : [a0] "v"(a[0]), [a1] "v"(a[1]), [a2] "v"(a[2]), [a3] "v"(a[3]), [xp] "v"(xp), [l] "i"(l));
}

// a[t] -= E(4 t + q, m) b for the lane's four rows, E(., m) by DPP from lane m
#define MPC_BLOCK_UPDATE(nop)                                                                 \
  asm(nop "v_fmac_f32_dpp %[a0], %[e0], -%[b]" MPC_NB                                         \
          "v_fmac_f32_dpp %[a1], %[e1], -%[b]" MPC_NB                                         \
          "v_fmac_f32_dpp %[a2], %[e2], -%[b]" MPC_NB                                         \
          "v_fmac_f32_dpp %[a3], %[e3], -%[b]" MPC_NB                                         \
      : [a0] "+v"(a[0]), [a1] "+v"(a[1]), [a2] "+v"(a[2]), [a3] "+v"(a[3])                    \
      : [e0] "v"(e[0]), [e1] "v"(e[1]), [e2] "v"(e[2]), [e3] "v"(e[3]), [b] "v"(b), [l] "i"(l))
template <int l>
__device__ __forceinline__ void block_update(float (&a)[4], const float (&e)[4], float b) {
  if constexpr (l == 0)
    MPC_BLOCK_UPDATE("s_nop 1\n");  // the wait states between the writes of e and their first DPP read
  else
    MPC_BLOCK_UPDATE("");
}
#undef MPC_BLOCK_UPDATE
template <int... M>
__device__ __forceinline__ void block_updates(float (&a)[4], const float (&e)[4], const float (&b)[NX],
                                              std::integer_sequence<int, M...>) {
  (block_update<M>(a, e, b[M]), ...);
}

// the quarters' lanes in scalar registers, and the ds_bpermute address of the
// lane's column in each quarter
struct Quarters {
  uint64_t mask[4];
  uint32_t from[4];
};

// Gauss-Jordan inverse of the block in a into x: pivot steps P .. 13.  rowa,
// rowx: row P of [A | X] in every quarter; piv, inv: its pivot and inverse;
// pivots: lane P holds pivot P.  DIV: inverses by division.
template <bool DIV, int P = 0>
__device__ __forceinline__ void gj_wave_steps(const Quarters &qs, float (&a)[4], float (&x)[4], float rowa, float rowx,
                                             float piv, float inv, float &pivots) {
  constexpr int QP = P & 3, TP = P >> 2;              // owner quarter and slot of row P
  asm("v_writelane_b32 %0, %1, %2" : "+v"(pivots) : "s"(piv), "i"(P));
  if constexpr (DIV) inv = 1.f / piv;
  const float ap = rowa * inv, xp = rowx * inv;
  if constexpr (P + 1 < NX) {
    constexpr int Q1 = (P + 1) & 3, T1 = (P + 1) >> 2;  // and of row P + 1
    const float next = pivot_first<DIV, P, 16 * Q1 + P + 1>(x[T1], a[T1], xp, ap);
    const float ra = lane_value(a[T1], qs.from[Q1]), rx = lane_value(x[T1], qs.from[Q1]);
    float ni;
    if constexpr (T1 == TP) {
      constexpr int o0 = T1 == 0 ? 1 : 0, o1 = T1 <= 1 ? 2 : 1, o2 = T1 <= 2 ? 3 : 2;
      ni = pivot_rest<P>(x[o0], a[o0], x[o1], a[o1], x[o2], a[o2], xp, ap, next, x[T1], a[T1], qs.mask[QP]);
    } else {
      constexpr int o1 = TP == 0 ? 2 : 0, o2 = TP <= 1 ? 3 : 1;
      static_assert(TP != T1 && o1 != TP && o2 != TP && o1 != T1 && o2 != T1 && o1 != o2, "the three other slots");
      ni = pivot_rest<P>(x[TP], a[TP], x[o1], a[o1], x[o2], a[o2], xp, ap, next, qs.mask[QP]);
    }
    gj_wave_steps<DIV, P + 1>(qs, a, x, ra, rx, next, ni, pivots);
  } else {
    pivot_last<P>(x, a, xp);
    const bool own = (qs.mask[QP] >> (threadIdx.x & 63u)) & 1u;
    x[TP] = own ? xp : x[TP];
  }
}

// base[off + c]: a lane's 32-bit element offset and a constant from a uniform base
__device__ __forceinline__ const float *at(const float *base, uint32_t off) {
  return reinterpret_cast<const float *>(reinterpret_cast<const char *>(base) + 4u * off);
}
__device__ __forceinline__ float *at(float *base, uint32_t off) {
  return reinterpret_cast<float *>(reinterpret_cast<char *>(base) + 4u * off);
}

template <bool TWO>
__device__ __forceinline__ void factor_wave(DirectLds<TWO> &lds, const float *__restrict__ S, float *work, const Pick &p,
                                           const Chain &ch, uint32_t lane) {
  FacWaveLds &L = lds.side[ch.side];
  const uint32_t q = lane >> 4, jl = lane & 15u, j = jl < (uint32_t)NX ? jl : NX - 1;
  const bool tail = q < 2u;  // slot 3 holds rows 12, 13 in quarters 0, 1
  Quarters qs;
  uint32_t rr[4], bl[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    qs.mask[t] = 0xFFFFull << (16 * t);
    qs.from[t] = 4u * (16u * t + jl);
    const uint32_t r = 4u * t + q, i = lane + 64u * t;
    rr[t] = r < (uint32_t)NX ? r : 0u;  // clamped row
    // place of element i of the block (side 1: transposed)
    const uint32_t br = ch.side ? i / NX : i % NX, bc = ch.side ? i % NX : i / NX;
    bl[t] = i < (uint32_t)NXX ? bc + RS * br : (uint32_t)(NX * RS) + jl;
  }
  const float *Sp = S + (size_t)S_STRIDE * p.K0;
  float *W = work + (size_t)S_STRIDE * p.K0;
  const uint32_t oa = NXX + q + NX * j, oe = q + NX * j;  // column j of a block from row q on, rows 4 apart
  // the knot's column elements and its B, read two knots ahead (what lies
  // past the block in its row is read with it and not used)
  float a_nxt[2][4], b_nxt[2][4];
  auto load = [&](float (&a)[4], float (&bb)[4], uint32_t k) {
    const uint32_t kc = k < ch.n ? k : ch.n;
    const float *Sd = Sp + (size_t)S_STRIDE * ch.knot(kc), *Sl = Sp + (size_t)S_STRIDE * ch.link(kc);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      a[t] = at(Sd, oa)[4 * t];
      bb[t] = at(Sl, lane)[64 * t];
    }
  };
  auto put_b = [&](const float (&bb)[4], uint32_t k) {
#pragma unroll
    for (int t = 0; t < 4; ++t) L.B[k & 1u][bl[t]] = -bb[t];
  };
  float a[4], x[4], b0[4];
  load(a, b0, 0);
  load(a_nxt[1], b_nxt[1], 1);
  load(a_nxt[0], b_nxt[0], 2);
  auto step = [&](uint32_t k, float (&an)[4], float (&bn)[4]) {
    float br[4][NX], bj[NX];
    float e[4] = {0.f, 0.f, 0.f, 0.f};
    if (k > 0) {
      // D_{k-1}^-1 from the quarters to columns
#pragma unroll
      for (int t = 0; t < 3; ++t) L.Dinv[4u * t + q + RS * j] = x[t];
      if (tail) L.Dinv[12u + q + RS * j] = x[3];
#pragma unroll
      for (int m = 0; m < NX; ++m) {
        bj[m] = L.B[k & 1u][m + RS * j];
#pragma unroll
        for (int t = 0; t < 4; ++t) br[t][m] = L.B[k & 1u][m + RS * rr[t]];
      }
      wave_sync();
      float dv[NX];
#pragma unroll
      for (int m = 0; m < NX; ++m) dv[m] = L.Dinv[m + RS * j];
#pragma unroll
      for (int t = 0; t < 4; ++t) a[t] = an[t];
      load(an, bn, k + 2);
      // E_b(r, j) = sum_m B(r, m) D_{b-1}^-1(m, j), m in order
#pragma unroll
      for (int m = 0; m < NX; ++m)
#pragma unroll
        for (int t = 0; t < 4; ++t) e[t] += br[t][m] * dv[m];
    }
    const bool meets = k == ch.n;
#pragma unroll
    for (int t = 0; t < 4; ++t) a[t] = (t < 3 || tail) && !(meets && ch.side) ? -a[t] : 0.f;
    // D_b(r, j) = A_b(r, j) - sum_m E(r, m) B(j, m), m in order
    if (k > 0) block_updates(a, e, bj, std::make_integer_sequence<int, NX>{});
    float *Wk = W + (size_t)S_STRIDE * ch.knot(k), *Wl = W + (size_t)S_STRIDE * ch.link(k);
    // lanes 14 and 15 store what lane 13 does
#pragma unroll
    for (int t = 0; t < 3; ++t) at(Wl, oe)[4 * t] = e[t];
    if (tail) at(Wl, oe)[12] = e[3];
    if (TWO && meets) {  // side 1's part to side 0, which inverts
      if (ch.side) {
#pragma unroll
        for (int t = 0; t < 4; ++t) lds.meet[t][lane] = a[t];
      }
      __syncthreads();
      if (ch.side) return;
#pragma unroll
      for (int t = 0; t < 4; ++t) a[t] += lds.meet[t][lane];
    }
    float keep[4], pivots = 1.f;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      keep[t] = a[t];
      x[t] = 4u * t + q == j ? 1.f : 0.f;
    }
    const float rowa = lane_value(a[0], qs.from[0]), rowx = j == 0 ? 1.f : 0.f, piv = read_lane<0>(a[0]);
    gj_wave_steps<false>(qs, a, x, rowa, rowx, piv, 1.f / piv, pivots);
    if (__builtin_amdgcn_ballot_w64(!mid_range(pivots)) != 0) {  // again, with divisions
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        a[t] = keep[t];
        x[t] = 4u * t + q == j ? 1.f : 0.f;
      }
      gj_wave_steps<true>(qs, a, x, rowa, rowx, piv, 1.f, pivots);
    }
#pragma unroll
    for (int t = 0; t < 3; ++t) at(Wk, oe)[NXX + 4 * t] = x[t];
    if (tail) at(Wk, oe)[NXX + 12] = x[3];
  };
  // B of the next knot goes to LDS ahead of the step that reads it
  put_b(b_nxt[1], 1);
  step(0, a_nxt[0], b_nxt[0]);
  for (uint32_t k = 1; k <= ch.n; k += 2) {
    put_b(b_nxt[0], k + 1);
    wave_sync();
    step(k, a_nxt[1], b_nxt[1]);
    if (k + 1 > ch.n) break;
    put_b(b_nxt[1], k + 2);
    wave_sync();
    step(k + 1, a_nxt[0], b_nxt[0]);
  }
}
#undef MPC_NB

// ---- substitution ------------------------------------------------------------
// The sweeps' chain is one 14-term dot product per knot (the terms by DPP
// row_newbcast in the multiply-adds, one after the other: about 70 clocks).
// The four rows of the wave hold the factor rows of four consecutive knots
// (so one set of reads serves four), and take their turns in the order 0, 1,
// 3, 2: from each to the next, and from the last to the first of the next
// four, the result moves by one lane swap.  What is off the chain (z_k =
// D_k^-1 y_k) runs once for the four knots.
// N = 256, both sweeps: 186 -> 49 us (before: one row, the vector by ds_swizzle).

// sum_m w[m] v_m, v_m the value v of lane m of the row (m < 14), in order
__device__ __forceinline__ float bdot(const float (&w)[NX], float v) {
  float s = 0.f;
#define MPC_BD(m, k) "v_fmac_f32_dpp %0, %1, %" #k " row_newbcast:" #m " row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
  asm("s_nop 1\n" MPC_BD(0, 2) MPC_BD(1, 3) MPC_BD(2, 4) MPC_BD(3, 5) MPC_BD(4, 6) MPC_BD(5, 7) MPC_BD(6, 8)
          MPC_BD(7, 9) MPC_BD(8, 10) MPC_BD(9, 11) MPC_BD(10, 12) MPC_BD(11, 13) MPC_BD(12, 14) MPC_BD(13, 15)
      : "+v"(s)
      : "v"(v), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "v"(w[4]), "v"(w[5]), "v"(w[6]), "v"(w[7]), "v"(w[8]),
        "v"(w[9]), "v"(w[10]), "v"(w[11]), "v"(w[12]), "v"(w[13]));
#undef MPC_BD
  return s;
}

// v of the row of turn s (rows 0, 1, 3, 2) in the row of the next turn:
// 0 -> 1 and 3 -> 2 by swapping neighbouring rows, 1 -> 3 and 2 -> 0 by
// swapping halves
template <int s>
__device__ __forceinline__ float pass_on(float v) {
  const uint32_t u = __builtin_bit_cast(uint32_t, v);
  uint32_t o;
  if constexpr (s & 1)
    o = __builtin_amdgcn_permlane32_swap(u, u, false, false)[s >> 1];
  else
    o = __builtin_amdgcn_permlane16_swap(u, u, false, false)[s >> 1];
  return __builtin_bit_cast(float, o);
}

// 14 consecutive floats at p, in pairs (a caller's workspace may lie at any
// multiple of four bytes, which 64-bit global reads take)
typedef float pair_u __attribute__((ext_vector_type(2), aligned(4)));
__device__ __forceinline__ void load14(float (&v)[NX], const float *p) {
  const pair_u *p2 = reinterpret_cast<const pair_u *>(p);
#pragma unroll
  for (int c = 0; c < NX / 2; ++c) {
    const pair_u t = p2[c];
    v[2 * c] = t.x;
    v[2 * c + 1] = t.y;
  }
}

// forward and backward sweeps of one side of an instance on the right-hand
// side r = -gamma, or with ACCUMULATE the workspace's z slots; lambda = x, or
// lambda += x with ACCUMULATE
template <bool TWO, bool ACCUMULATE>
__device__ __forceinline__ void substitute(DirectLds<TWO> &lds, const float *__restrict__ gamma, float *work,
                                          float *__restrict__ lambda, const Pick &p, const Chain &ch, uint32_t lane) {
  const uint32_t q = lane >> 4, i = lane & 15u, j = i < (uint32_t)NX ? i : NX - 1;
  const uint32_t turn = q ^ (q >> 1);  // rows 0, 1, 3, 2 in order
  const bool el = i < (uint32_t)NX;
  float *W = work + (size_t)S_STRIDE * p.K0, *lp = lambda + (size_t)NX * p.K0;
  const float *gp = ACCUMULATE ? nullptr : gamma + (size_t)NX * p.K0;
  // positions k0 .. k0 + 3 of the forward sweep, position k0 + turn in the row
  // (the meeting knot's data again past it): row j of E_k (strided; E_0 = 0),
  // row j of D_k^-1 (= column j, D^-1 symmetric) and the right-hand side (the
  // meeting knot's on side 0 alone)
  struct Fwd {
    float er[NX], dr[NX], r;
  };
  auto load_f = [&](Fwd &f, uint32_t k0) {
    const uint32_t k = k0 + turn < ch.n ? k0 + turn : ch.n;
    const float *E = at(W, S_STRIDE * ch.link(k) + j);
#pragma unroll
    for (int m = 0; m < NX; ++m) f.er[m] = E[NX * m];
    const uint32_t kn = ch.knot(k);
    load14(f.dr, at(W, S_STRIDE * kn + NX * j) + NXX);
    const float r = ACCUMULATE ? at(W, S_STRIDE * kn + j)[2 * NXX] : -*at(gp, NX * kn + j);
    f.r = ch.side && k == ch.n ? 0.f : r;
  };
  float y = 0.f, yo = 0.f;
  auto run_f = [&](const Fwd &f, uint32_t k0) {
    float t;  // yo: the row's own y
    t = f.r - bdot(f.er, y);
    yo = t;
    y = pass_on<0>(t);
    if (k0 + 1 <= ch.n) {
      t = f.r - bdot(f.er, y);
      yo = turn == 1u ? t : yo;
      y = pass_on<1>(t);
    }
    if (k0 + 2 <= ch.n) {
      t = f.r - bdot(f.er, y);
      yo = turn == 2u ? t : yo;
      y = pass_on<2>(t);
    }
    if (k0 + 3 <= ch.n) {
      t = f.r - bdot(f.er, y);
      yo = turn == 3u ? t : yo;
      y = pass_on<3>(t);
    }
    const float z = bdot(f.dr, yo);
    if (el && k0 + turn < ch.n) *at(W, S_STRIDE * ch.knot(k0 + turn) + 2 * NXX + i) = z;
  };
  Fwd f[3];
#pragma unroll
  for (int u = 0; u < 3; ++u) load_f(f[u], 4u * u);
  for (uint32_t k0 = 0; k0 <= ch.n; k0 += 12) {
#pragma unroll
    for (int u = 0; u < 3; ++u) {
      const uint32_t k = k0 + 4u * u;
      if (k > ch.n) break;
      run_f(f[u], k);
      load_f(f[u], k + 12u);
    }
  }
  // the meeting knot: y = side 0's + side 1's part, x = D^-1 y
  const uint32_t km = chain_of<TWO>(p.N, 0).n;
  const bool owner = turn == (ch.n & 3u);  // the row whose turn it was last
  if (ch.side && owner) lds.v[i] = yo;
  __syncthreads();  // (z, read by other lanes below, too)
  if (!ch.side) {
    float dr[NX];
    load14(dr, at(W, S_STRIDE * km + NX * j) + NXX);
    const float l = ACCUMULATE ? *at(lp, NX * km + j) : 0.f;
    if (owner) lds.x[i] = TWO ? yo + lds.v[i] : yo;
    wave_sync();
    const float xm = bdot(dr, lds.x[j]);
    wave_sync();
    if (q == 0) lds.x[i] = xm;
    if (el && q == 0) *at(lp, NX * km + i) = ACCUMULATE ? l + xm : xm;
  }
  __syncthreads();
  // backward: position top - turn in the row (position 0 again past the
  // start): column j of E_{k+1}, z_k and the value that x_k is added to
  struct Bwd {
    float ec[NX], z, l;
  };
  auto load_b = [&](Bwd &g, int top) {
    const uint32_t k = top - (int)turn > 0 ? (uint32_t)(top - (int)turn) : 0u;
    load14(g.ec, at(W, S_STRIDE * ch.link(k < ch.n ? k + 1u : ch.n) + NX * j));
    const uint32_t kn = ch.knot(k);
    g.z = *at(W, S_STRIDE * kn + 2 * NXX + j);
    g.l = ACCUMULATE ? *at(lp, NX * kn + j) : 0.f;
  };
  float x = lds.x[j];
  auto run_b = [&](const Bwd &g, int top) {
    float xo, t;
    t = g.z - bdot(g.ec, x);
    xo = t;
    x = pass_on<0>(t);
    if (top >= 1) {
      t = g.z - bdot(g.ec, x);
      xo = turn == 1u ? t : xo;
      x = pass_on<1>(t);
    }
    if (top >= 2) {
      t = g.z - bdot(g.ec, x);
      xo = turn == 2u ? t : xo;
      x = pass_on<2>(t);
    }
    if (top >= 3) {
      t = g.z - bdot(g.ec, x);
      xo = turn == 3u ? t : xo;
      x = pass_on<3>(t);
    }
    if (el && top >= (int)turn) *at(lp, NX * ch.knot((uint32_t)(top - (int)turn)) + i) = ACCUMULATE ? g.l + xo : xo;
  };
  Bwd g[3];
  const int n = (int)ch.n;
#pragma unroll
  for (int u = 0; u < 3; ++u) load_b(g[u], n - 1 - 4 * u);
  for (int top0 = n - 1; top0 >= 0; top0 -= 12) {
#pragma unroll
    for (int u = 0; u < 3; ++u) {
      const int top = top0 - 4 * u;
      if (top < 0) break;
      run_b(g[u], top);
      load_b(g[u], top - 12);
    }
  }
}

// one workgroup per instance, a wave per side: the factorisation (FACTOR;
// else the factors a previous launch left in work), then the substitution
// sweeps on r = -gamma, or with ACCUMULATE on the z slots, added to lambda
template <bool TWO, bool FACTOR, bool ACCUMULATE>
__global__ void __launch_bounds__(TWO ? 128 : 64) k_direct_wave(Batch b, const uint32_t *__restrict__ order,
                                                    const float *__restrict__ S, const float *__restrict__ gamma,
                                                    const uint32_t *__restrict__ status, float *work,
                                                    float *__restrict__ lambda, uint32_t *__restrict__ iters,
                                                    uint32_t *__restrict__ flag) {
  __shared__ DirectLds<TWO> lds;
  const uint32_t lane = threadIdx.x & 63u;
  const Pick p = pick_instance(b, order, status, blockIdx.x);
  if (!p.live) return;
  const Chain ch = chain_of<TWO>(p.N, TWO ? (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) : 0u);
  if constexpr (FACTOR) {
    factor_wave<TWO>(lds, S, work, p, ch, lane);
    __syncthreads();  // the factor rows written above are read below
  }
  substitute<TWO, ACCUMULATE>(lds, gamma, work, lambda, p, ch, lane);
  if (!ACCUMULATE && threadIdx.x == 0) {
    if (iters) iters[p.inst] = 0;
    if (flag) flag[p.inst] = 0;
  }
}

// z slot of every knot <- -gamma + S lambda (fp64 accumulation), one group per knot
__global__ void __launch_bounds__(WG) k_schur_residual(Batch b, const float *__restrict__ S,
                                                       const float *__restrict__ gamma,
                                                       const float *__restrict__ lambda, float *__restrict__ work) {
  const int grp = threadIdx.x / GROUP, lane = threadIdx.x % GROUP;
  const uint32_t gk = blockIdx.x * GROUPS_PER_WG + grp;
  if (gk >= b.total_knots || lane >= NX) return;
  const KnotRef kr = locate(b, gk);
  const float *Sr = S + (size_t)S_STRIDE * gk;
  const float *l = lambda + (size_t)NX * gk;
  double res = -(double)gamma[(size_t)NX * gk + lane];
#pragma unroll
  for (int m = 0; m < NX; ++m) res += (double)Sr[NXX + lane + NX * m] * (double)l[m];
  if (kr.k > 0) {
#pragma unroll
    for (int m = 0; m < NX; ++m) res += (double)Sr[lane + NX * m] * (double)l[m - NX];
  }
  if (kr.k + 1 < kr.N) {  // S(b,b+1) = S(b+1,b)^T: the next block row's left block
#pragma unroll
    for (int m = 0; m < NX; ++m) res += (double)Sr[S_STRIDE + m + NX * lane] * (double)l[m + NX];
  }
  slot_z(work, gk)[lane] = (float)res;
}

}  // namespace

template <bool TWO>
static hipError_t direct_solve(const Batch &b, const uint32_t *order, uint32_t n_list, const float *S,
                               const float *gamma, const uint32_t *status, float *work, float *lambda,
                               uint32_t steps, bool do_factor, uint32_t *iters, uint32_t *flag, hipStream_t st) {
  const dim3 grid(n_list), block(TWO ? 128 : 64);
  if (do_factor)
    hipLaunchKernelGGL((k_direct_wave<TWO, true, false>), grid, block, 0, st, b, order, S, gamma, status, work, lambda,
                       iters, flag);
  else
    hipLaunchKernelGGL((k_direct_wave<TWO, false, false>), grid, block, 0, st, b, order, S, gamma, status, work,
                       lambda, iters, flag);
  hipError_t e = hipGetLastError();
  for (uint32_t s = 0; s < steps && e == hipSuccess; ++s) {
    hipLaunchKernelGGL(k_schur_residual, dim3((b.total_knots + GROUPS_PER_WG - 1) / GROUPS_PER_WG), dim3(WG), 0, st,
                       b, S, gamma, (const float *)lambda, work);
    e = hipGetLastError();
    if (e != hipSuccess) break;
    hipLaunchKernelGGL((k_direct_wave<TWO, false, true>), grid, block, 0, st, b, order, S, gamma, status, work, lambda,
                       (uint32_t *)nullptr, (uint32_t *)nullptr);
    e = hipGetLastError();
  }
  return e;
}

// Both ends at once take one refinement step more than asked.  The two orders
// of elimination round differently, by up to the error of an unrefined solve
// (5e-4 relative at N = 256) or of one refined twice (1e-6; 3e-8, the rounding
// of lambda itself, on well-conditioned systems): after the same number of
// steps either may be the closer one (over 324 systems, N = 2 .. 512, R =
// 1e-2 .. 1e-6, rho 1e-3 and 1, two steps: by up to 20 and 14 times).  With the
// step more that the halved chains pay for, both ends at once were at least as
// close on every one.  So the caller must have asked for two steps; with fewer
// it is one order, that of the knots, and its bits.
// It pays while the longest chain lasts longer than the work of all knots spread
// over half the device's SIMDs (for equal horizons: two instances per compute
// unit, a SIMD for each of their waves).  Two refinement steps from one end /
// from both, us: N = 64, 1 instance 139 / 101, 256 158 / 129, 512 185 / 181, past the
// line 1024 272 / 286, 4096 878 / 1116; N = 256, 1 490 / 322, 256 564 / 420, 512 714 /
// 710, 1024 1145 / 1261, 2048 2022 / 2461; N = 16, 51 / 48, 54 / 53, 62 / 66, 90 / 92, 4096
// 216 / 271; N = 32 .. 512 mixed, 512 instances 1149 / 879, 1024 1349 / 1250, past
// the line (from 1187 on) 1280 1456 / 1450, 2048 1850 / 2122.
bool direct_both_ends(uint32_t n_cu, uint32_t total_knots, uint32_t longest, uint32_t refine) {
  return refine >= 2 && total_knots <= 2ull * n_cu * longest;
}

hipError_t launch_direct_solve(const Batch &b, const uint32_t *order, uint32_t n_list, const float *S,
                               const float *gamma, const uint32_t *status, float *work, float *lambda,
                               uint32_t refine, bool both_ends, bool do_factor, uint32_t *iters, uint32_t *flag,
                               hipStream_t st) {
  if (n_list == 0) return hipSuccess;
  return both_ends ? direct_solve<true>(b, order, n_list, S, gamma, status, work, lambda, refine + 1u, do_factor,
                                        iters, flag, st)
                   : direct_solve<false>(b, order, n_list, S, gamma, status, work, lambda, refine, do_factor, iters,
                                         flag, st);
}

}  // namespace mpc
