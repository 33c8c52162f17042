// k_pcg_split.hip -- block-Jacobi PCG in split-preconditioned form for
// gfx950: one 512-lane workgroup per bin of instances (N <= 256 each).
//
// Block-Jacobi PCG on S lambda = gamma (preconditioner Pinv = S(b,b)^-1) is,
// in exact arithmetic, plain CG on the transformed system
//     S^ lambda^ = gamma^,  S^ = W^T S W,  gamma^ = W^T gamma,  lambda = W lambda^,
// with W = diag(W_b), W_b = U_b^-1 and -S(b,b) = theta_b = U_b^T U_b
// (Cholesky).  S^ has -I on its diagonal and L^_b = W_b^T S(b,b-1) W_{b-1}
// below it; the preconditioner becomes -I, and the residuals satisfy
// r^ = W^T r, so r^T z^ = r^T Pinv r: the exit test |r^T z| < tol and every
// alpha, beta are those of the reference's PCG (GPU-PCG pcg<T,14,N>, call site
// toplevel.cuh:143-157), and the iterates map to its iterates.  Only L^ is
// kept on chip (one 14 x 14 block per knot instead of S(b,b), Pinv(b,b) and
// S(b,b-1)), and an iteration takes two block products instead of four.
//
// k_split_prep forms L^_b, W_b and gamma^_b from S and gamma (one 16-lane
// group per knot, W_b by Gauss elimination of theta_b without pivoting:
// theta is symmetric positive definite); k_pcg_split runs the iteration.
//
// Layout of the split system (the Pinv buffer's rows): L^_b at offset 0 of
// row b, W_b at offset NXX (both 14 x 14, column-major), gamma^ in its own
// buffer.
//
// Workgroup: 32 groups of 16 lanes (8 waves), group g serving knots
// 8g .. 8g+7 of its instance, lane i element i; up to 256 knots, bins of
// up to 8 instances, each on whole waves (as in pcg_res_body.h).  The
// blocks are held pre-rotated for the DPP products of pcg_onchip.h, in
// registers and LDS slots of the group's own (below).
#include "common.h"
#include "gj16.h"
#include "pcg_onchip.h"

namespace mpc {

namespace {

using namespace onchip;

constexpr int GROUP = 16;

// ---------------------------------------------------------------- prep ----
// Workgroups of PG groups overlap by one knot: group g of workgroup w serves
// row kg = (PG - 1) w + g - 1.  Every group forms W of its row; groups
// g >= 1 then take W of the row before from group g - 1 through LDS.
constexpr int PG = 16;
constexpr int PWG = PG * GROUP;

struct alignas(16) PrepLds {
  float W[NXX];  // W_kg, column-major
  float L[NXX];  // S(kg, kg-1), column-major
  float gm[16];
};

__global__ void __launch_bounds__(PWG) k_split_prep(Batch b, const float *__restrict__ S,
                                                    const float *__restrict__ gamma,
                                                    const uint32_t *__restrict__ status, float *__restrict__ Ps,
                                                    float *__restrict__ ghat) {
  __shared__ PrepLds lds[PG];
  const int grp = threadIdx.x / GROUP, lane = threadIdx.x % GROUP;
  const int64_t kg_raw = (int64_t)blockIdx.x * (PG - 1) + grp - 1;
  const bool in_range = kg_raw >= 0 && kg_raw < (int64_t)b.total_knots;
  const uint32_t kg = in_range ? (uint32_t)kg_raw : 0u;
  const KnotRef kr = locate(b, kg);
  const bool active = in_range && !(status && !(status[kr.inst] & ST_ACTIVE));
  const bool owner = grp > 0 && active;
  PrepLds &L = lds[grp];
  const int j = lane < NX ? lane : NX - 1;
  const float *Sr = S + (size_t)S_STRIDE * kg;
  // 1. theta = -S(kg,kg) by columns; W_kg = chol(theta)^-1 by rows
  float a[NX], x[NX];
#pragma unroll
  for (int r = 0; r < NX; ++r) a[r] = -Sr[NXX + r + NX * j];
  chol_inv_rows<NX>(lane, a, x);
  // x[c] = W^T(c, j) = W(j, c): lane j holds row j of W
  if (lane < NX) {
#pragma unroll
    for (int c = 0; c < NX; ++c) L.W[lane + NX * c] = x[c];
  }
  const bool row0 = kr.k == 0;
  for (int i = lane; i < NXX; i += GROUP) L.L[i] = row0 ? 0.f : Sr[i];
  if (lane < NX) L.gm[lane] = gamma[(size_t)NX * kg + lane];
  __syncthreads();
  // 2. row kg: M = S(kg,kg-1) W_{kg-1} (column j per lane), L^ = W_kg^T M,
  //    gamma^ = W_kg^T gamma_kg
  float *Pr = Ps + (size_t)S_STRIDE * kg;
  if (owner) {
    const PrepLds &Pv = lds[grp - 1];
    float m[NX];
#pragma unroll
    for (int r = 0; r < NX; ++r) m[r] = 0.f;
    if (!row0) {
#pragma unroll
      for (int k = 0; k < NX; ++k) {
        const float wkj = Pv.W[k + NX * j];
#pragma unroll
        for (int r = 0; r < NX; ++r) m[r] += L.L[r + NX * k] * wkj;
      }
    }
    float lh[NX];
#pragma unroll
    for (int r = 0; r < NX; ++r) {
      float acc = 0.f;
#pragma unroll
      for (int k = 0; k < NX; ++k) acc += L.W[k + NX * r] * m[k];
      lh[r] = acc;
    }
    if (lane < NX) {
#pragma unroll
      for (int r = 0; r < NX; ++r) Pr[r + NX * lane] = lh[r];
      float gacc = 0.f;
#pragma unroll
      for (int k = 0; k < NX; ++k) gacc += L.W[k + NX * lane] * L.gm[k];
      ghat[(size_t)NX * kg + lane] = gacc;
    }
    for (int i = lane; i < NXX; i += GROUP) Pr[NXX + i] = L.W[i];
  }
}

// --------------------------------------------------------------- solve ----
// One 512-lane workgroup (8 waves, two per SIMD, up to 256 VGPRs each) per
// bin: 32 groups of 16 lanes, group g serving knots 8g .. 8g+7 of its
// instance.  A block L^_b enters two products per iteration, L^_b x_{b-1}
// and L^_b^T x_b.  Held as rotated rows (Mr[n] = L(i, src(i, n))) the first
// is 16 multiply-adds with the vector rotated by DPP; held as rotated rows of
// its transpose (Kr[n] = L(src(i, n), i)) so is the second.  From rows
// alone the transposed product needs the products rotated instead (Horner
// form: 16 products and 15 rotated additions).  Per group, of the nine
// blocks L^_{8g} .. L^_{8g+8} (the last is the next group's first):
//   registers: rows of L^_1 .. L^_7, transposed rows of L^_3 and L^_4;
//   LDS slots: rows of L^_0, transposed rows of L^_1, L^_2 and L^_8;
// so L^_5 .. L^_7 take the Horner form.  Two 16-register buffers take the
// slot reads, each issued one product group ahead of its use, and the
// products run as four or five interleaved chains: with two waves per SIMD
// a wave's own independent instructions hide the latency of the chains.
constexpr int NT = 512;
constexpr int NGRP = NT / 16;     // 32 groups
constexpr int RK = 8;             // knots per group
constexpr int KNOTS = NGRP * RK;  // 256
constexpr int MAXI = 8;  // instances per bin (act is read as two 16-byte words)

// A block slot: rotated row element n of lane i at ((n >> 1) * 16 + i) * 2 +
// (n & 1), read as 8 x 64-bit words (each 16-lane read covers the 32 banks
// once); lanes 14, 15 hold zeros.
constexpr int SLOT = 256;

struct SplitShared {
  float R0[NGRP * SLOT];     // rows of L^_{8g}
  float K1[NGRP * SLOT];     // rows of L^_{8g+1}^T
  float K2[NGRP * SLOT];     // rows of L^_{8g+2}^T
  float K8[NGRP * SLOT];     // rows of L^_{8g+8}^T
  float zb[NGRP * 2 * 16 + 16];  // staged vector element of each group's first and last knot, then zeros
  float red[2][MAXI][NGRP];  // dot-product partials: one per group, by instance and group
  uint32_t act[MAXI];        // by instance of the bin: 1 while it iterates
};
constexpr uint32_t SPLIT_CLEAR4 = (uint32_t)(sizeof(SplitShared) / 16);
static_assert(sizeof(SplitShared) % 16 == 0 && offsetof(SplitShared, act) % 16 == 0, "cleared and read as 16-byte words");

__device__ __forceinline__ void write_slot(float *Sl, uint32_t i, const float (&M)[16]) {
  float2 *s2 = reinterpret_cast<float2 *>(Sl) + i;
#pragma unroll
  for (int c = 0; c < 8; ++c) s2[16 * c] = make_float2(M[2 * c], M[2 * c + 1]);
}

__device__ __forceinline__ void read_slot(float (&M)[16], const float *Sl, uint32_t i) {
  const float2 *s2 = reinterpret_cast<const float2 *>(Sl) + i;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const float2 v = s2[16 * c];
    M[2 * c] = v.x;
    M[2 * c + 1] = v.y;
  }
}

// (M_k^T x_k)_i for three blocks with rotated rows M_k: sum_n ror_n(m_n),
// m_n = M[(16 - n) & 15] x, in Horner form m_0 + ror_1(m_1 + ror_1(m_2 + ...
// + ror_1(m_15))): 16 products and 15 row_ror:1 additions per block, the
// three chains interleaved.  A DPP instruction needs two wait states after
// the VALU write of what it reads; per step the three products come first,
// then the three additions, so the distances are there without an s_nop
// (the compiler's order, product and addition of one chain back to back,
// put one ahead of each of the 45 additions: 8.3 clocks an instruction of a
// lone wave against 4.7).
#define MPC_HSTEP(m0, m1, m2)                                                                           \
  "v_mul_f32 %3, %" #m0 ", %6\n"                                                                        \
  "v_mul_f32 %4, %" #m1 ", %7\n"                                                                        \
  "v_mul_f32 %5, %" #m2 ", %8\n"                                                                        \
  "v_add_f32_dpp %0, %0, %3 row_ror:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n"                        \
  "v_add_f32_dpp %1, %1, %4 row_ror:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n"                        \
  "v_add_f32_dpp %2, %2, %5 row_ror:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
#define MPC_HORNER3(k0, k1, k2)                                                                         \
  asm(MPC_HSTEP(9, 10, 11) MPC_HSTEP(12, 13, 14) MPC_HSTEP(15, 16, 17)                                  \
      : "+v"(a0), "+v"(a1), "+v"(a2), "=&v"(t0), "=&v"(t1), "=&v"(t2)                                   \
      : "v"(x0), "v"(x1), "v"(x2), "v"(M0[k0]), "v"(M1[k0]), "v"(M2[k0]), "v"(M0[k1]), "v"(M1[k1]),     \
        "v"(M2[k1]), "v"(M0[k2]), "v"(M1[k2]), "v"(M2[k2]))
__device__ __forceinline__ void rot_mtv3(const float (&M0)[16], float x0, const float (&M1)[16], float x1,
                                         const float (&M2)[16], float x2, float &c0, float &c1, float &c2) {
  float a0 = M0[1] * x0, a1 = M1[1] * x1, a2 = M2[1] * x2, t0, t1, t2;
  MPC_HORNER3(2, 3, 4);
  MPC_HORNER3(5, 6, 7);
  MPC_HORNER3(8, 9, 10);
  MPC_HORNER3(11, 12, 13);
  MPC_HORNER3(14, 15, 0);
  c0 = a0;
  c1 = a1;
  c2 = a2;
}
#undef MPC_HORNER3
#undef MPC_HSTEP

// two blocks of rot_mtv3
#define MPC_HSTEP(m0, m1)                                                        \
  "v_mul_f32 %2, %" #m0 ", %4\n"                                                 \
  "v_mul_f32 %3, %" #m1 ", %5\n"                                                 \
  "v_add_f32_dpp %0, %0, %2 row_ror:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n" \
  "v_add_f32_dpp %1, %1, %3 row_ror:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
#define MPC_HORNER2(k0, k1, k2)                                                                        \
  asm(MPC_HSTEP(6, 7) MPC_HSTEP(8, 9) MPC_HSTEP(10, 11)                                                  \
      : "+v"(a0), "+v"(a1), "=&v"(t0), "=&v"(t1)                                                        \
      : "v"(x0), "v"(x1), "v"(M0[k0]), "v"(M1[k0]), "v"(M0[k1]), "v"(M1[k1]), "v"(M0[k2]), "v"(M1[k2]))
__device__ __forceinline__ void rot_mtv2(const float (&M0)[16], float x0, const float (&M1)[16], float x1, float &c0,
                                         float &c1) {
  float a0 = M0[1] * x0, a1 = M1[1] * x1, t0, t1;
  MPC_HORNER2(2, 3, 4);
  MPC_HORNER2(5, 6, 7);
  MPC_HORNER2(8, 9, 10);
  MPC_HORNER2(11, 12, 13);
  MPC_HORNER2(14, 15, 0);
  c0 = a0;
  c1 = a1;
}
#undef MPC_HORNER2
#undef MPC_HSTEP

// Three to five interleaved accumulations a_k += sum_{n=1..15} M_k[n] * ror_n(x_k),
// three terms per asm statement; an s_nop ahead of the first (the two wait
// states between a VALU write of x_k and its DPP read; that no copy of x_k lands
// right ahead of a later one is checked by tests/test_wait_states.py)
#define MPC_TERM(n, acc, x, m) \
  "v_fmac_f32_dpp %" #acc ", %" #x ", %" #m " row_ror:" #n " row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
#define MPC_T4(n, m0, m1, m2, m3) MPC_TERM(n, 0, 4, m0) MPC_TERM(n, 1, 5, m1) MPC_TERM(n, 2, 6, m2) MPC_TERM(n, 3, 7, m3)
#define MPC_B4(pre, n0, n1, n2)                                                                                 \
  asm(pre MPC_T4(n0, 8, 9, 10, 11) MPC_T4(n1, 12, 13, 14, 15) MPC_T4(n2, 16, 17, 18, 19)                        \
      : "+v"(a), "+v"(b), "+v"(c), "+v"(e)                                                                     \
      : "v"(xa), "v"(xb), "v"(xc), "v"(xe), "v"(Ma[n0]), "v"(Mb[n0]), "v"(Mc[n0]), "v"(Me[n0]), "v"(Ma[n1]),     \
        "v"(Mb[n1]), "v"(Mc[n1]), "v"(Me[n1]), "v"(Ma[n2]), "v"(Mb[n2]), "v"(Mc[n2]), "v"(Me[n2]))
__device__ __forceinline__ void rot_fma15x4(float &a, float xa, const float (&Ma)[16], float &b, float xb,
                                            const float (&Mb)[16], float &c, float xc, const float (&Mc)[16],
                                            float &e, float xe, const float (&Me)[16]) {
  MPC_B4("s_nop 1\n", 1, 2, 3);
  MPC_B4("", 4, 5, 6);
  MPC_B4("", 7, 8, 9);
  MPC_B4("", 10, 11, 12);
  MPC_B4("", 13, 14, 15);
}
#undef MPC_B4
#undef MPC_T4
#define MPC_T3(n, m0, m1, m2) MPC_TERM(n, 0, 3, m0) MPC_TERM(n, 1, 4, m1) MPC_TERM(n, 2, 5, m2)
#define MPC_B3(pre, n0, n1, n2)                                                                               \
  asm(pre MPC_T3(n0, 6, 7, 8) MPC_T3(n1, 9, 10, 11) MPC_T3(n2, 12, 13, 14)                                      \
      : "+v"(a), "+v"(b), "+v"(c)                                                                               \
      : "v"(xa), "v"(xb), "v"(xc), "v"(Ma[n0]), "v"(Mb[n0]), "v"(Mc[n0]), "v"(Ma[n1]), "v"(Mb[n1]), "v"(Mc[n1]), \
        "v"(Ma[n2]), "v"(Mb[n2]), "v"(Mc[n2]))
__device__ __forceinline__ void rot_fma15x3(float &a, float xa, const float (&Ma)[16], float &b, float xb,
                                            const float (&Mb)[16], float &c, float xc, const float (&Mc)[16]) {
  MPC_B3("s_nop 1\n", 1, 2, 3);
  MPC_B3("", 4, 5, 6);
  MPC_B3("", 7, 8, 9);
  MPC_B3("", 10, 11, 12);
  MPC_B3("", 13, 14, 15);
}
#undef MPC_B3
#undef MPC_T3
#define MPC_T5(n, m0, m1, m2, m3, m4) \
  MPC_TERM(n, 0, 5, m0) MPC_TERM(n, 1, 6, m1) MPC_TERM(n, 2, 7, m2) MPC_TERM(n, 3, 8, m3) MPC_TERM(n, 4, 9, m4)
#define MPC_B5(pre, n0, n1, n2)                                                                                  \
  asm(pre MPC_T5(n0, 10, 11, 12, 13, 14) MPC_T5(n1, 15, 16, 17, 18, 19) MPC_T5(n2, 20, 21, 22, 23, 24)          \
      : "+v"(a), "+v"(b), "+v"(c), "+v"(e), "+v"(f)                                                             \
      : "v"(xa), "v"(xb), "v"(xc), "v"(xe), "v"(xf), "v"(Ma[n0]), "v"(Mb[n0]), "v"(Mc[n0]), "v"(Me[n0]),        \
        "v"(Mf[n0]), "v"(Ma[n1]), "v"(Mb[n1]), "v"(Mc[n1]), "v"(Me[n1]), "v"(Mf[n1]), "v"(Ma[n2]), "v"(Mb[n2]), \
        "v"(Mc[n2]), "v"(Me[n2]), "v"(Mf[n2]))
__device__ __forceinline__ void rot_fma15x5(float &a, float xa, const float (&Ma)[16], float &b, float xb,
                                            const float (&Mb)[16], float &c, float xc, const float (&Mc)[16],
                                            float &e, float xe, const float (&Me)[16], float &f, float xf,
                                            const float (&Mf)[16]) {
  MPC_B5("s_nop 1\n", 1, 2, 3);
  MPC_B5("", 4, 5, 6);
  MPC_B5("", 7, 8, 9);
  MPC_B5("", 10, 11, 12);
  MPC_B5("", 13, 14, 15);
}
#undef MPC_B5
#undef MPC_T5
#undef MPC_TERM

// base[off], with a 32-bit byte offset from a uniform base (one address
// register; an instance's rows are at most 256 * 2352 bytes)
__device__ __forceinline__ float at(const float *__restrict__ base, uint32_t off) {
  return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(base) + 4u * off);
}

// element offsets of the rotated rows of a block of row b0
__device__ __forceinline__ void block_offsets(uint32_t (&off)[16], uint32_t b0, uint32_t i, uint32_t d) {
#pragma unroll
  for (int n = 0; n < 16; ++n) {
    const uint32_t j = (i + (uint32_t)n * d) & 15u;
    off[n] = S_STRIDE * b0 + i + (j < (uint32_t)NX ? NX * j : 0u);
  }
}

// Rotated rows of a column-major 14 x 14 block (its element (i, src(i, n)) at
// base + off[n], i = the lane), zeros where ok is false; one branch for the
// block's 16 reads, none between them.
__device__ __forceinline__ void load_lrows(float (&Lr)[16], bool ok, uint32_t i, uint32_t d, const float *__restrict__ base,
                                           const uint32_t (&off)[16]) {
#pragma unroll
  for (int n = 0; n < 16; ++n) Lr[n] = 0.f;
  if (ok) {
#pragma unroll
    for (int n = 0; n < 16; ++n) Lr[n] = at(base, off[n]);
#pragma unroll
    for (int n = 0; n < 16; ++n) Lr[n] = ((i + (uint32_t)n * d) & 15u) < (uint32_t)NX ? Lr[n] : 0.f;
  }
}

// the slot of the block's transpose from its rotated rows: the element of
// lane i, rotation n is the one of lane src(i, n), rotation -n, there
__device__ __forceinline__ void write_slot_t(float *Sl, uint32_t i, uint32_t d, const float (&M)[16]) {
#pragma unroll
  for (int n = 0; n < 16; ++n) {
    const uint32_t m = (16u - (uint32_t)n) & 15u, c = (i + (uint32_t)n * d) & 15u;
    Sl[((m >> 1) * 16u + c) * 2u + (m & 1u)] = M[n];
  }
}

__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_pcg_split(Batch b, const uint4 *__restrict__ items, const uint32_t *__restrict__ bin_off,
            const float *__restrict__ Ps, const float *__restrict__ ghat, float *__restrict__ lambda,
            uint32_t max_iter, float tol, const uint32_t *__restrict__ status, uint32_t *__restrict__ iters_out,
            uint32_t *__restrict__ flag_out, float *__restrict__ eta_out) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  SplitShared &sh = *reinterpret_cast<SplitShared *>(smem_raw);
  const uint32_t tid = threadIdx.x, bin = blockIdx.x;
  const uint32_t g = tid >> 4, i = tid & 15u;
  const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t d = ror_step(tid);
  {
    float4 *z4 = reinterpret_cast<float4 *>(smem_raw);
    for (uint32_t idx = tid; idx < SPLIT_CLEAR4; idx += NT) z4[idx] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  // the wave's instance in this bin (items: {inst, first group, groups, -};
  // an instance owns whole waves, so everything about it is uniform over the
  // wave and stays in scalar registers)
  const uint32_t i0 = bin_off[bin], ni = bin_off[bin + 1] - i0;
  int slot = -1;
  uint32_t inst = 0, g0 = 0;
  for (uint32_t jx = 0; jx < ni; ++jx) {
    const uint4 it = items[i0 + jx];
    if (4u * w >= it.y && 4u * w < it.y + it.z) {
      slot = (int)jx;
      inst = it.x;
      g0 = it.y;
    }
  }
  const bool mine = slot >= 0;
  const uint32_t N = mine ? inst_len(b, inst) : 0u;
  const uint32_t K0 = mine ? inst_first(b, inst) : 0u;
  const bool live = uniform(mine && !(status && !(status[inst] & ST_ACTIVE)));
  const uint32_t cap = pcg_cap(max_iter, N);
  const uint32_t lg = g - g0;
  const bool lane_ok = i < (uint32_t)NX;
  __syncthreads();  // LDS cleared

  // ---- load: lambda^ = W^-1 lambda by back substitution (W upper
  // triangular) and gamma^, then the blocks (fewer values live at once).
  // The reads of a wave that has no instance, or of knots past its end, go
  // to a valid row (clamped) and are replaced by zeros.
  const uint32_t b0 = lg * RK;
  const float *Pw = Ps + (size_t)S_STRIDE * K0;  // the instance's rows
  const uint32_t klast = N ? N - 1u : 0u, il = lane_ok ? i : 0u;
  auto knot = [&](uint32_t t) { return b0 + t < klast ? b0 + t : klast; };
  float lam[RK], r[RK], p[RK], y[RK];  // z = -r is not stored; r starts as gamma^
  bool any = false;
#pragma unroll
  for (int t = 0; t < RK; ++t) {
    const bool has = live && b0 + (uint32_t)t < N && lane_ok;
    const float l = lambda[(size_t)NX * (K0 + knot(t)) + il], h = ghat[(size_t)NX * (K0 + knot(t)) + il];
    lam[t] = has ? l : 0.f;
    r[t] = has ? h : 0.f;
    any = any || lam[t] != 0.f;
  }
  // A start from lambda = 0 has lambda^ = 0.  Otherwise the group's eight
  // back substitutions run in lockstep: in step k lane t of the row takes
  // knot t's pivot quotient (from lane k of that knot, by DPP), so one
  // division serves all eight, and each goes back to its row by DPP.
  if (__builtin_amdgcn_ballot_w64(any) != 0) {
    float wr[RK][NX], den[NX];
    const uint32_t td = i & (RK - 1);
#pragma unroll
    for (int k = 0; k < NX; ++k) {
      const float v = at(Pw, S_STRIDE * knot(td) + NXX + k + NX * k);
      den[k] = live ? v : 1.f;
    }
#pragma unroll
    for (int t = 0; t < RK; ++t)
#pragma unroll
      for (int c = 0; c < NX; ++c) wr[t][c] = at(Pw, S_STRIDE * knot(t) + NXX + il + NX * c);
    float lh[RK];
#pragma unroll
    for (int t = 0; t < RK; ++t) lh[t] = 0.f;
#pragma unroll
    for (int k = NX - 1; k >= 0; --k) {
      float num = 0.f;
#pragma unroll
      for (int t = 0; t < RK; ++t) {
        const float v = bcast_dyn16(lam[t], k);
        num = td == (uint32_t)t ? v : num;
      }
      const float quo = num / den[k];
#pragma unroll
      for (int t = 0; t < RK; ++t) {
        const float xk = bcast_dyn16(quo, t);
        lh[t] = (int)i == k ? xk : lh[t];
        lam[t] -= wr[t][k] * xk;
      }
      pin(lh);
      pin(lam);
    }
#pragma unroll
    for (int t = 0; t < RK; ++t) lam[t] = live && b0 + (uint32_t)t < N && lane_ok ? lh[t] : 0.f;
  }
  asm volatile("" ::: "memory");  // the block reads below stay behind the rows of W
  float *R0g = sh.R0 + g * SLOT, *K1g = sh.K1 + g * SLOT, *K2g = sh.K2 + g * SLOT, *K8g = sh.K8 + g * SLOT;
  auto ok = [&](uint32_t t) { return live && lane_ok && b0 + t < N && b0 + t > 0; };  // L^_0 = 0
  uint32_t roff[16];
  block_offsets(roff, b0, i, d);
  // Only rows are read (a group's 16 reads of a block touch its 784 bytes
  // once each; reading the transposes by lanes 56 bytes apart took 36 k
  // clocks of address processing for a full workgroup); the transposes are
  // written from them, through the slot of L^_0 where they end in registers.
  float Lr[RK - 1][16];  // Lr[t - 1]: rows of L^_t, t = 1 .. 7
  float Kr[2][16];       // Kr[t - 3]: rows of L^_t^T, t = 3, 4
#pragma unroll
  for (int t = 1; t < RK; ++t) load_lrows(Lr[t - 1], ok(t), i, d, Pw + S_STRIDE * t, roff);
  write_slot_t(K1g, i, d, Lr[0]);
  write_slot_t(K2g, i, d, Lr[1]);
#pragma unroll
  for (int t = 3; t < 5; ++t) {
    write_slot_t(R0g, i, d, Lr[t - 1]);
    wave_sync();
    read_slot(Kr[t - 3], R0g, i);
    wave_sync();
  }
  {
    float Ls[16];
    load_lrows(Ls, ok(RK), i, d, Pw + S_STRIDE * RK, roff);
    write_slot_t(K8g, i, d, Ls);
    load_lrows(Ls, ok(0), i, d, Pw, roff);
    write_slot(R0g, i, Ls);
  }
  // zb: [group][first, last knot][lane]; a group without a neighbour reads
  // the zero entries behind the last group's
  float *zbg = sh.zb + g * 32 + i;
  const float *zm_src = lg > 0 ? zbg - 16 : sh.zb + NGRP * 32 + i, *zp_src = b0 + RK < N ? zbg + 32 : sh.zb + NGRP * 32 + i;
  auto stage = [&](const float (&v)[RK]) {
    zbg[0] = v[0];
    zbg[16] = v[RK - 1];
  };
  auto stage_neg = [&](const float (&v)[RK]) {
    zbg[0] = -v[0];
    zbg[16] = -v[RK - 1];
  };
  // y = S^ x: y_t = -x_t + L^_t x_{t-1} + L^_{t+1}^T x_{t+1}; xm / xp: the
  // elements of knots 8lg - 1 and 8lg + 8.  Lanes 14, 15 of every block row
  // are zero, so y (and r, p, lambda^) stay zero there.
  // two slot buffers: each slot read is issued one product group ahead of
  // its use; A holds the rows of L^_0 between calls
  float A[16], B[16];
  read_slot(A, R0g, i);
  auto smv = [&](const float (&x)[RK], float xm, float xp) {
    read_slot(B, K1g, i);
    // first chain of every knot: rows of L^_t times x_{t-1}
    y[0] = fmaf(A[0], xm, -x[0]);
#pragma unroll
    for (int t = 1; t < 5; ++t) y[t] = fmaf(Lr[t - 1][0], x[t - 1], -x[t]);
    rot_fma15x5(y[0], xm, A, y[1], x[0], Lr[0], y[2], x[1], Lr[1], y[3], x[2], Lr[2], y[4], x[3], Lr[3]);
    read_slot(A, K2g, i);
#pragma unroll
    for (int t = 5; t < 8; ++t) y[t] = fmaf(Lr[t - 1][0], x[t - 1], -x[t]);
    y[0] = fmaf(B[0], x[1], y[0]);
    rot_fma15x4(y[5], x[4], Lr[4], y[6], x[5], Lr[5], y[7], x[6], Lr[6], y[0], x[1], B);
    read_slot(B, K8g, i);
    float c4, c5, c6;
    rot_mtv3(Lr[4], x[5], Lr[5], x[6], Lr[6], x[7], c4, c5, c6);
    // second chains: rows of L^_{t+1}^T times x_{t+1}
    y[1] = fmaf(A[0], x[2], y[1]);
    y[2] = fmaf(Kr[0][0], x[3], y[2]);
    y[3] = fmaf(Kr[1][0], x[4], y[3]);
    y[7] = fmaf(B[0], xp, y[7]);
    rot_fma15x4(y[1], x[2], A, y[2], x[3], Kr[0], y[3], x[4], Kr[1], y[7], xp, B);
    read_slot(A, R0g, i);
    y[4] += c4;
    y[5] += c5;
    y[6] += c6;
  };
  // dot products: a row total per group to LDS (red[k][instance][group]),
  // then, after the barrier, the instance's 32 entries (zero past its
  // groups) summed by every row: two per lane, then the row total
  float *redg = &sh.red[0][mine ? slot : 0][lg & (NGRP - 1)];
  auto post = [&](int k, float part) {
    const float v = row_total(part);
    redg[k * MAXI * NGRP] = v;  // the row's lanes write the same value
  };
  const float2 *red2 = reinterpret_cast<const float2 *>(&sh.red[0][mine ? slot : 0][0]) + i;
  auto total = [&](int k) {
    const float2 v = red2[k * MAXI * NGRP / 2];
    return row_total(v.x + v.y);
  };
  stage(lam);
  // an instance's act word: set here, cleared when it stops (its lanes all
  // write the same, between the second barrier of its last iteration and the
  // first of the next)
  if (live) sh.act[slot] = 1u;
  __syncthreads();
  float pm = *zm_src, pp = *zp_src;

  // The first pass is the prologue, through the same code (one copy of the
  // products): p = lambda^, r = gamma^ - S^ lambda^ (alpha = 1, lambda^ kept),
  // z = -r, then p = z (beta = 0) and eta = r.z; the others are the
  // iterations.  The loop has no branch on a value that differs between
  // lanes (one would put every branch of it on EXEC masks, several hundred
  // clocks of mask bookkeeping per iteration) and none but its own for a wave
  // that iterates.
#pragma unroll
  for (int t = 0; t < RK; ++t) p[t] = lam[t];
  uint32_t it = ~0u;  // the first pass is not counted
  float eta = 0.f, tol_i = tol;
  bool conv = !live;
  if (live) {
    bool first = true, run;
    do {
      smv(p, pm, pp);
      float pyp = 0.f;
#pragma unroll
      for (int t = 0; t < RK; ++t) pyp += p[t] * y[t];
      post(0, pyp);
      __syncthreads();
      const float quo = eta / total(0), alpha = first ? 1.f : quo;
      float rz = 0.f;
#pragma unroll
      for (int t = 0; t < RK; ++t) {
        r[t] -= alpha * y[t];
        rz -= r[t] * r[t];
      }
      stage_neg(r);
      post(1, rz);
      __syncthreads();
      const float zm = *zm_src, zp = *zp_src, eta_new = total(1);
      const float alpha_l = first ? 0.f : alpha;
#pragma unroll
      for (int t = 0; t < RK; ++t) lam[t] += alpha_l * p[t];
      // taken in the last iteration too (p is not used after it)
      const float quo_b = eta_new / eta, beta = first ? 0.f : quo_b;
      eta = eta_new;
#pragma unroll
      for (int t = 0; t < RK; ++t) p[t] = fmaf(beta, p[t], -r[t]);
      pm = fmaf(beta, pm, zm);
      pp = fmaf(beta, pp, zp);
      // tol < 0: exit relative to the first residual, |eta| < -tol |eta_0|
      if (first && tol < 0.f) tol_i = fmaxf(-tol * fabsf(eta), FLT_MIN);
      ++it;
      first = false;
      conv = uniform(fabsf(eta) < tol_i);  // eta is the same in every lane
      run = !conv && it < cap;
    } while (run);
    sh.act[slot] = 0u;
  }
  // Waves that iterate no more (or have no instance) keep the others'
  // barriers until no instance of the bin iterates.  They read the act words
  // between the two barriers, where those do not change, so all leave in the
  // same round.
  for (;;) {
    __syncthreads();
    const uint4 a0 = reinterpret_cast<const uint4 *>(sh.act)[0], a1 = reinterpret_cast<const uint4 *>(sh.act)[1];
    if (uniform((a0.x | a0.y | a0.z | a0.w | a1.x | a1.y | a1.z | a1.w) == 0u)) break;
    __syncthreads();
  }

  if (!live) return;
  // lambda = W lambda^, two knots at a time (the offsets formed again, not
  // held through the iterations)
  uint32_t ie = i;
  asm volatile("" : "+v"(ie));
  uint32_t woff[16];
  block_offsets(woff, b0, ie, d);
#pragma unroll
  for (int t = 0; t < RK; t += 2) {
    float Wr[2][16];
#pragma unroll
    for (int u = 0; u < 2; ++u)
      load_lrows(Wr[u], lane_ok && b0 + (uint32_t)(t + u) < N, i, d, Pw + S_STRIDE * (t + u) + NXX, woff);
    float va, vb;
    rot_mv2(Wr[0], lam[t], va, Wr[1], lam[t + 1], vb);
    if (b0 + t < N && lane_ok) lambda[(size_t)NX * (K0 + b0 + t) + i] = va;
    if (b0 + t + 1 < N && lane_ok) lambda[(size_t)NX * (K0 + b0 + t + 1) + i] = vb;
  }
  if (lg == 0 && i == 0) {
    if (iters_out) iters_out[inst] = it;
    if (flag_out) flag_out[inst] = conv ? 0u : 1u;
    if (eta_out) eta_out[inst] = fabsf(eta);
  }
}

// ------------------------------------------------- short instances ----
// A few short instances (N <= 64), a workgroup of up to four waves each: the
// iteration above with the eight knots of a group on two 16-lane rows, four
// each, so that twice the SIMDs share the products.  Bitwise the same, so each
// knot keeps the form of its second product (L^_5 .. L^_7 the Horner form), and
// a slot whose two rows differ in it takes both.  With knots 0, 1, 4, 5 on the
// even row and 2, 3, 6, 7 on the odd one that is one slot of the four:
//   slot  knot (even, odd row)  first product  second product
//   0     0, 2                  rows L^_t      transposed rows L^_{t+1}
//   1     1, 3                  rows L^_t      transposed rows L^_{t+1}
//   2     4, 6                  rows L^_t      Horner from the rows L^_{t+1} (slot 3's)
//   3     5, 7                  rows L^_t      even: Horner from rows, odd: transposed rows
// All blocks are in registers, neighbours on the other row come by lane swaps,
// and the group's sums pass from row to row in the knots' order.  The group's
// outer neighbour is knot 8g - 1 for the even row and 8g + 8 for the odd one.
// Iterations of N = 64 take 0.92 us against 1.17 (173 of them on a device of
// 256 instances 238 -> 187 us), the layer's solves of 256 instances 594 -> 471
// us on average.
constexpr int SH_RK = 4;  // knots per row

constexpr int SH_NT = 256;               // four waves
constexpr int SH_KNOTS = 64;
constexpr int SH_GRP = SH_KNOTS / RK;    // groups of eight knots

struct ShortShared {
  float slot[SH_NT / 16 * SLOT];         // a block per row, to transpose it
  float zb[(SH_GRP + 2) * 2 * 16];       // staged first and last knot of group + 1, zeros at both ends
  alignas(16) float red[2][2 * SH_GRP];  // group sums; the second half takes the writes of the even rows
};

// u of the even rows and v of the even rows | u of the odd rows and v of the
// odd rows, in the even | odd rows
__device__ __forceinline__ void swap16(float u, float v, float &evens, float &odds) {
  const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, u), __builtin_bit_cast(uint32_t, v),
                                                  false, false);
  evens = __builtin_bit_cast(float, (uint32_t)r[0]);
  odds = __builtin_bit_cast(float, (uint32_t)r[1]);
}

__global__ void __launch_bounds__(SH_NT) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_pcg_split_short(Batch b, const float *__restrict__ Ps, const float *__restrict__ ghat, float *__restrict__ lambda,
                  uint32_t max_iter, float tol, const uint32_t *__restrict__ status, uint32_t *__restrict__ iters_out,
                  uint32_t *__restrict__ flag_out, float *__restrict__ eta_out) {
  __shared__ ShortShared sh;
  const uint32_t tid = threadIdx.x, inst = blockIdx.x;
  const uint32_t i = tid & 15u, row = tid >> 4, g = tid >> 5;
  const bool odd = row & 1u;
  const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t d = ror_step(tid);
  for (uint32_t k = tid; k < (SH_GRP + 2) * 2 * 16; k += SH_NT) sh.zb[k] = 0.f;
  if (tid < 4u * SH_GRP) (&sh.red[0][0])[tid] = 0.f;
  const uint32_t N = inst_len(b, inst), K0 = inst_first(b, inst);
  if (status && !(status[inst] & ST_ACTIVE)) return;
  __syncthreads();  // LDS cleared
  if (16u * w >= N) return;  // no knots: the other waves' barriers go on without this one
  const uint32_t cap = pcg_cap(max_iter, N);
  const bool lane_ok = i < (uint32_t)NX;

  // the slots' knots
  const uint32_t t0 = RK * g + (odd ? 2u : 0u);
  auto knot = [&](int t) { return t0 + (uint32_t)(t & 1) + (t & 2 ? 4u : 0u); };
  const float *Pw = Ps + (size_t)S_STRIDE * K0;  // the instance's rows
  const uint32_t il = lane_ok ? i : 0u;
  auto clamped = [&](int t) { return knot(t) < N ? knot(t) : N - 1u; };
  float lam[SH_RK], r[SH_RK], p[SH_RK], y[SH_RK];
  bool any = false;
#pragma unroll
  for (int t = 0; t < SH_RK; ++t) {
    const bool has = knot(t) < N && lane_ok;
    const float l = lambda[(size_t)NX * (K0 + clamped(t)) + il], h = ghat[(size_t)NX * (K0 + clamped(t)) + il];
    lam[t] = has ? l : 0.f;
    r[t] = has ? h : 0.f;
    any = any || lam[t] != 0.f;
  }
  // lambda^ = W^-1 lambda by back substitution, four knots in lockstep (above)
  if (__builtin_amdgcn_ballot_w64(any) != 0) {
    float wr[SH_RK][NX], den[NX], lh[SH_RK];
    const uint32_t td = i & (SH_RK - 1);
    const uint32_t kd = t0 + (td & 1u) + (td & 2u ? 4u : 0u);
#pragma unroll
    for (int k = 0; k < NX; ++k) den[k] = at(Pw, S_STRIDE * (kd < N ? kd : N - 1u) + NXX + k + NX * k);
#pragma unroll
    for (int t = 0; t < SH_RK; ++t) {
      lh[t] = 0.f;
#pragma unroll
      for (int c = 0; c < NX; ++c) wr[t][c] = at(Pw, S_STRIDE * clamped(t) + NXX + il + NX * c);
    }
#pragma unroll
    for (int k = NX - 1; k >= 0; --k) {
      float num = 0.f;
#pragma unroll
      for (int t = 0; t < SH_RK; ++t) {
        const float v = bcast_dyn16(lam[t], k);
        num = td == (uint32_t)t ? v : num;
      }
      const float quo = num / den[k];
#pragma unroll
      for (int t = 0; t < SH_RK; ++t) {
        const float xk = bcast_dyn16(quo, t);
        lh[t] = (int)i == k ? xk : lh[t];
        lam[t] -= wr[t][k] * xk;
      }
      pin(lh);
      pin(lam);
    }
#pragma unroll
    for (int t = 0; t < SH_RK; ++t) lam[t] = knot(t) < N && lane_ok ? lh[t] : 0.f;
  }
  asm volatile("" ::: "memory");  // the block reads below stay behind the rows of W
  // the rows of L^ of the slots' knots; transposed through the row's LDS slot
  // those of the knot after slots 0 and 1 and, odd rows, after slot 3 (even
  // rows hold its rows there)
  float L[SH_RK][16], K0r[16], K1r[16], Z[16];
  uint32_t roff[16];
  block_offsets(roff, t0, i, d);
  auto block = [&](float (&M)[16], uint32_t dk) {  // rows of L^_{t0 + dk}, L^_0 = 0
    load_lrows(M, lane_ok && t0 + dk < N && t0 + dk > 0u, i, d, Pw + S_STRIDE * dk, roff);
  };
  float *mine = sh.slot + row * SLOT;
  auto transpose = [&](float (&M)[16], const float (&A)[16]) {
    write_slot_t(mine, i, d, A);
    wave_sync();
    read_slot(M, mine, i);
    wave_sync();
  };
  block(L[0], 0);
  block(L[1], 1);
  block(L[2], 4);
  block(L[3], 5);
  block(Z, 6);
  transpose(K0r, L[1]);
  {
    float A[16];
    block(A, 2);
    transpose(K1r, A);
    transpose(A, Z);
#pragma unroll
    for (int n = 0; n < 16; ++n) Z[n] = odd ? A[n] : Z[n];
  }

  float *zs = sh.zb + (g + 1u) * 32u + (odd ? 16u : 0u) + i;
  const float *zn_src = sh.zb + (odd ? (g + 2u) * 32u : g * 32u + 16u) + i;
  auto smv = [&](float pn) {
    float x0p, x1n, x2p, x3n, e, o;
    swap16(pn, p[1], x0p, o);
    swap16(p[0], p[2], e, o);
    x1n = odd ? e : o;
    swap16(p[1], p[3], e, o);
    x2p = odd ? e : o;
    swap16(p[2], pn, e, x3n);
    y[0] = fmaf(L[0][0], x0p, -p[0]);
    y[1] = fmaf(L[1][0], p[0], -p[1]);
    y[2] = fmaf(L[2][0], x2p, -p[2]);
    y[3] = fmaf(L[3][0], p[2], -p[3]);
    rot_fma15x4(y[0], x0p, L[0], y[1], p[0], L[1], y[2], x2p, L[2], y[3], p[2], L[3]);
    float yd = fmaf(Z[0], x3n, y[3]), c2, c3;
    y[0] = fmaf(K0r[0], p[1], y[0]);
    y[1] = fmaf(K1r[0], x1n, y[1]);
    rot_fma15x3(y[0], p[1], K0r, y[1], x1n, K1r, yd, x3n, Z);
    rot_mtv2(L[3], p[3], Z, x3n, c2, c3);
    y[2] += c2;
    c3 = y[3] + c3;
    y[3] = odd ? yd : c3;
  };
  // sum over the group's eight knots of u v in their order, in the odd row
  auto group_dot = [&](const float (&u)[SH_RK], const float (&v)[SH_RK], bool neg) {
    auto add = [&](float s, int t) { return fmaf(neg ? -u[t] : u[t], v[t], s); };
    float s, e, o;
    s = add(add(0.f, 0), 1);
    swap16(s, s, s, o);   // knots 0, 1 to the odd row
    s = add(add(s, 0), 1);
    swap16(s, s, e, s);   // .. 3 to the even one
    s = add(add(s, 2), 3);
    swap16(s, s, s, o);
    return add(add(s, 2), 3);
  };
  float *red_dst = &sh.red[0][odd ? g : SH_GRP + g];
  auto post = [&](int k, float s) { red_dst[k * 2 * SH_GRP] = row_total(s); };
  // in the order of the kernel above: pairs, then the levels of row_total
  // (past the eight groups it adds zeros)
  static_assert(SH_GRP == 8, "eight group sums");
  auto total = [&](int k) {
    const float4 a = *reinterpret_cast<const float4 *>(&sh.red[k][0]), c = *reinterpret_cast<const float4 *>(&sh.red[k][4]);
    return (((a.x + a.y) + (a.z + a.w)) + ((c.x + c.y) + (c.z + c.w))) + 0.f;
  };
  *zs = odd ? lam[3] : lam[0];
  __syncthreads();
  float pn = *zn_src;
  // (the iteration as above)
#pragma unroll
  for (int t = 0; t < SH_RK; ++t) p[t] = lam[t];
  uint32_t it = ~0u;  // the first pass is not counted
  float eta = 0.f, tol_i = tol;
  bool first = true, conv, run;
  do {
    smv(pn);
    post(0, group_dot(p, y, false));
    __syncthreads();
    const float quo = eta / total(0), alpha = first ? 1.f : quo;
#pragma unroll
    for (int t = 0; t < SH_RK; ++t) r[t] -= alpha * y[t];
    *zs = odd ? -r[3] : -r[0];
    post(1, group_dot(r, r, true));
    __syncthreads();
    const float zn = *zn_src, eta_new = total(1);
    const float alpha_l = first ? 0.f : alpha;
#pragma unroll
    for (int t = 0; t < SH_RK; ++t) lam[t] += alpha_l * p[t];
    // taken in the last iteration too (p is not used after it)
    const float quo_b = eta_new / eta, beta = first ? 0.f : quo_b;
    eta = eta_new;
#pragma unroll
    for (int t = 0; t < SH_RK; ++t) p[t] = fmaf(beta, p[t], -r[t]);
    pn = fmaf(beta, pn, zn);
    if (first && tol < 0.f) tol_i = fmaxf(-tol * fabsf(eta), FLT_MIN);
    ++it;
    first = false;
    conv = uniform(fabsf(eta) < tol_i);  // eta is the same in every lane
    run = !conv && it < cap;
  } while (run);

  // lambda = W lambda^, two knots at a time
  uint32_t ie = i;
  asm volatile("" : "+v"(ie));
  uint32_t woff[16];
  block_offsets(woff, t0, ie, d);
#pragma unroll
  for (int t = 0; t < SH_RK; t += 2) {
    float Wr[2][16], v[2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
      load_lrows(Wr[u], lane_ok && knot(t + u) < N, i, d, Pw + S_STRIDE * (2 * t + u) + NXX, woff);
    rot_mv2(Wr[0], lam[t], v[0], Wr[1], lam[t + 1], v[1]);
#pragma unroll
    for (int u = 0; u < 2; ++u)
      if (knot(t + u) < N && lane_ok) lambda[(size_t)NX * (K0 + knot(t + u)) + i] = v[u];
  }
  if (tid == 0) {
    if (iters_out) iters_out[inst] = it;
    if (flag_out) flag_out[inst] = conv ? 0u : 1u;
    if (eta_out) eta_out[inst] = fabsf(eta);
  }
}

}  // namespace

uint32_t pcg_split_max_knots() { return (uint32_t)KNOTS; }
uint32_t pcg_split_bin_groups() { return (uint32_t)NGRP; }
uint32_t pcg_split_max_items() { return (uint32_t)MAXI; }
uint32_t pcg_split_groups(uint32_t N) {
  const uint32_t groups = (N + RK - 1) / RK;
  return (groups + 3u) & ~3u;  // whole waves
}

hipError_t launch_split_prep(const Batch &b, const float *S, const float *gamma, const uint32_t *status, float *Ps,
                             float *ghat, hipStream_t st) {
  if (b.total_knots == 0) return hipSuccess;
  const dim3 grid((b.total_knots + PG - 2) / (PG - 1));
  hipLaunchKernelGGL(k_split_prep, grid, dim3(PWG), 0, st, b, S, gamma, status, Ps, ghat);
  return hipGetLastError();
}

hipError_t launch_pcg_split(const Batch &b, const uint4 *items, const uint32_t *bin_off, uint32_t n_bins,
                            const float *Ps, const float *ghat, float *lambda, uint32_t max_iter, float tol,
                            const uint32_t *status, uint32_t *iters, uint32_t *flag, float *eta, hipStream_t st) {
  if (n_bins == 0) return hipSuccess;
  static bool attr_set = false;
  const size_t smem = sizeof(SplitShared);
  if (!attr_set) {
    (void)hipFuncSetAttribute((const void *)k_pcg_split, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    (void)hipGetLastError();
    attr_set = true;
  }
  hipLaunchKernelGGL(k_pcg_split, dim3(n_bins), dim3(NT), smem, st, b, items, bin_off, Ps, ghat, lambda, max_iter,
                     tol, status, iters, flag, eta);
  return hipGetLastError();
}

uint32_t pcg_split_short_knots() { return (uint32_t)SH_KNOTS; }

hipError_t launch_pcg_split_short(const Batch &b, uint32_t n_inst, const float *Ps, const float *ghat, float *lambda,
                                  uint32_t max_iter, float tol, const uint32_t *status, uint32_t *iters,
                                  uint32_t *flag, float *eta, hipStream_t st) {
  if (n_inst == 0) return hipSuccess;
  hipLaunchKernelGGL(k_pcg_split_short, dim3(n_inst), dim3(SH_NT), 0, st, b, Ps, ghat, lambda, max_iter, tol, status,
                     iters, flag, eta);
  return hipGetLastError();
}

}  // namespace mpc
