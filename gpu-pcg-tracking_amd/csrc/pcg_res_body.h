// pcg_res_body.h -- the workgroup body of the resident on-chip PCG
// (gfx950), shared by its own kernel (k_pcg_res.hip) and the mixed
// cooperative launch that runs bins beside teams (k_pcg_team.hip).
//
// Same algorithm and exit rule as k_pcg.hip (GPU-PCG pcg<T,14,N>, call
// site toplevel.cuh:143-157), but every instance's matrix is read from HBM
// once per solve, and vectors never leave registers except for one
// neighbour exchange per iteration (block-row arithmetic: pcg_onchip.h).
//
// A 512-lane workgroup holds up to 128 knots: 32 groups of 16 lanes, each
// serving RK = 4 consecutive knots (4 lg + t of its instance, t = 0..3); a
// 256-lane one holds 64 knots, and two of them share a CU.
// Several instances share a workgroup ("bin"): each owns whole waves, so
// its dot products are a wave64 reduction plus a fixed-order sum over its
// own waves, and its arithmetic does not depend on which bin it is packed
// into.  Instances of a bin iterate in lockstep; a converged instance
// skips its arithmetic until the bin is done.
//
// With the stair preconditioner (STAIR), z = D^-1 (2 r - S D^-1 r): one more
// block product, one more staged vector and one more barrier per iteration.
//
// Per iteration, two workgroup barriers (block Jacobi):
//   y = S p; p.y -> B1 -> alpha; lambda, r;
//   z = Pinv r; stage z of the group's first and last knot; r.z -> B2 ->
//   beta; p = z + beta p for the own knots and, from the staged z, for the
//   copies of the neighbouring groups' elements p_{4lg-1}[i], p_{4lg+4}[i]
//   (the same fused multiply-add as their owners, so every copy stays
//   bitwise equal to its owner).
// The two waves of a SIMD issue their products one after the other (a DPP
// multiply-add takes 4.5 clocks, a plain one 2.25), so the iteration is bound
// by issue; branches on values that differ between lanes cost it several
// hundred clocks in EXEC bookkeeping, so conditions are ballots and the loop
// has one back branch.  Batch of 300 in stair mode 5.34 -> 3.98 ms, 3.73 with
// S(b,b-1) in registers too (it was read from LDS twice per product); one
// stair solve of N = 100 1.46 -> 1.15 ms.
#pragma once
#include "pcg_onchip.h"

namespace mpc {
namespace resident {

using namespace onchip;

constexpr int RK = 4;    // knots per group
constexpr int MAXI = 8;  // instances per bin

// Workgroup shapes: NT = 512 lanes (32 groups, 8 waves, 128 knots; one per
// CU) or 256 (16 groups, 4 waves, 64 knots; two per CU).
template <int NT>
struct ResShape {
  static_assert(NT == 256 || NT == 512, "workgroup of 4 or 8 waves");
  static constexpr int NGRP = NT / 16, NWAV = NT / 64, KNOTS = NGRP * RK;
};

template <int NT>
struct ResShared {
  static constexpr int KNOTS = ResShape<NT>::KNOTS, NWAV = ResShape<NT>::NWAV;
  float zb[(KNOTS + 1) * 16];  // staged vector element per knot slot and lane (+ one zero slot)
  float wb[(KNOTS + 1) * 16];  // stair preconditioner: staged D^-1 r
  // dot-product partials of the waves, by instance of the bin and wave of the
  // instance (zero past its waves)
  alignas(16) float red[2][MAXI][NWAV];
  uint32_t act[MAXI];  // by instance of the bin: 1 while it iterates
  static_assert(NWAV % 4 == 0, "partials are read as 16-byte words");
};

// the partials in wave order
template <int NWAV>
__device__ __forceinline__ float seg_sum(const float (&red)[NWAV]) {
  float s = 0.f;
#pragma unroll
  for (int v = 0; v < NWAV; v += 4) {
    const float4 x = *reinterpret_cast<const float4 *>(red + v);
    s = (((s + x.x) + x.y) + x.z) + x.w;
  }
  return s;
}

// The PCG of bin `bin` (its instances: items[bin_off[bin] .. bin_off[bin+1]))
// on an NT-lane workgroup with the ResShared<NT> block at smem; tid is
// threadIdx.x (passed in so that a caller's loop can keep everything
// derived from it inside the loop).
template <bool STAIR, int NT>
__device__ __forceinline__ void body(uint32_t tid, uint32_t bin, unsigned char *smem, Batch b,
                                     const uint4 *__restrict__ items,
                                     const uint32_t *__restrict__ bin_off, const float *__restrict__ S,
                                     const float *__restrict__ Pinv, const float *__restrict__ gamma,
                                     float *__restrict__ lambda, uint32_t max_iter, float tol,
                                     const uint32_t *__restrict__ status, uint32_t *__restrict__ iters_out,
                                     uint32_t *__restrict__ flag_out, float *__restrict__ eta_out) {
  constexpr int NWAV = ResShape<NT>::NWAV, KNOTS = ResShape<NT>::KNOTS;
  ResShared<NT> &sh = *reinterpret_cast<ResShared<NT> *>(smem);
  const uint32_t g = tid >> 4, i = tid & 15u, w = tid >> 6;
  const uint32_t d = ror_step(tid);
  for (uint32_t idx = tid; idx < (KNOTS + 1) * 16; idx += NT) sh.zb[idx] = 0.f;

  // my instance in this bin (items: {inst, first group, groups, -}); a null
  // item table means one instance (0) starting at group 0
  uint32_t i0 = 0, ni = 1;
  if (items) {
    i0 = bin_off[bin];
    ni = bin_off[bin + 1] - i0;
  }
  // (whole waves per instance: everything about it is uniform over the wave)
  const uint32_t ws = (uint32_t)__builtin_amdgcn_readfirstlane((int)w);
  int slot = -1;
  uint32_t inst = 0, g0 = 0;
  const uint32_t ng1 = ((inst_len(b, 0) + RK - 1) / RK + 3u) & ~3u;  // lone instance: as in a bin
  for (uint32_t j = 0; j < ni; ++j) {
    const uint4 it = items ? items[i0 + j] : make_uint4(0u, 0u, ng1, 0u);
    if (4u * ws >= it.y && 4u * ws < it.y + it.z) {
      slot = (int)j;
      inst = it.x;
      g0 = it.y;
    }
  }
  const bool mine = slot >= 0;
  const uint32_t N = mine ? inst_len(b, inst) : 0u;
  const uint32_t K0 = mine ? inst_first(b, inst) : 0u;
  const bool live = uniform(mine && !(status && !(status[inst] & ST_ACTIVE)));
  const uint32_t cap = pcg_cap(max_iter, N);
  const uint32_t lg = g - g0, lbase = g0 * RK;
  const bool lane_ok = i < (uint32_t)NX;
  if (tid < (uint32_t)MAXI) sh.act[tid] = 0u;
  if (tid < 2u * MAXI * NWAV) (&sh.red[0][0][0])[tid] = 0.f;
  __syncthreads();  // LDS cleared

  // ---- load: the block rows
  const uint32_t b0 = lg * RK, s0 = lbase + b0;  // first knot of the group and its slot
  Rows<RK> R;
  R.load(S + (size_t)S_STRIDE * K0, Pinv + (size_t)S_STRIDE * K0, b0, live ? N : 0u, N, i, d);
  float lam[RK], r[RK], p[RK], y[RK], z[RK];
#pragma unroll
  for (int t = 0; t < RK; ++t) {
    const uint32_t bk = b0 + (uint32_t)t;
    const bool has = live && bk < N && lane_ok;
    lam[t] = has ? lambda[(size_t)NX * (K0 + bk) + i] : 0.f;
    r[t] = has ? gamma[(size_t)NX * (K0 + bk) + i] : 0.f;
  }
  // first / last element of the group to LDS; neighbouring groups' copies back
  const bool in_m = lg > 0, in_p = b0 + RK < N;
  float *zb0 = sh.zb + s0 * 16 + i;
  auto stage = [&](const float (&v)[RK]) {
    zb0[0] = v[0];
    zb0[(RK - 1) * 16] = v[RK - 1];
  };
  // (the last knot's slot is followed by a zero one, and the first reads it)
  const float *zm_src = in_m ? zb0 - 16 : sh.zb + KNOTS * 16 + i, *zp_src = in_p ? zb0 + RK * 16 : sh.zb + KNOTS * 16 + i;
  auto neighbours = [&](float &vm, float &vp) {
    vm = *zm_src;
    vp = *zp_src;
  };
  // stair preconditioner: the first / last element of w = D^-1 r, the same way
  float *wb0 = sh.wb + s0 * 16 + i;
  auto stage_w = [&](const float (&v)[RK]) {
    wb0[0] = v[0];
    wb0[(RK - 1) * 16] = v[RK - 1];
  };
  const float *wm_src = in_m ? wb0 - 16 : sh.zb + KNOTS * 16 + i, *wp_src = in_p ? wb0 + RK * 16 : sh.zb + KNOTS * 16 + i;
  auto neighbours_w = [&](float &vm, float &vp) {
    vm = *wm_src;
    vp = *wp_src;
  };
  // y = S x for the group's knots; xm / xp: elements of knots 4lg-1, 4lg+4
  auto smv = [&](const float (&x)[RK], float xm, float xp) { group_smv<RK>(R, x, xm, xp, y); };
  // an instance's act word: set here, cleared when it stops (its lanes all
  // write the same, between the second barrier of its last iteration and the
  // first of the next)
  if (live) sh.act[slot] = 1u;
  stage(lam);
  __syncthreads();
  float pm, pp;
  neighbours(pm, pp);

  // The first pass is the prologue, through the same code: p = lambda,
  // r = gamma - S lambda (alpha = 1, lambda kept), z = M r, then p = z
  // (beta = 0) and eta = r.z; the others are the iterations.  The loop's
  // only branch is its own, on a scalar condition: with more the compiler
  // puts all of them on EXEC masks (its divergent stores are none of them).
#pragma unroll
  for (int t = 0; t < RK; ++t) p[t] = lam[t];
  uint32_t it = ~0u;  // the first pass is not counted
  float eta = 0.f, tol_i = tol;
  bool conv = !live;
  if (live) {
    float(&red0)[NWAV] = sh.red[0][slot], (&red1)[NWAV] = sh.red[1][slot];
    const uint32_t wi = ws - (g0 >> 2);  // wave of the instance
    bool first = true, run;
    do {
      smv(p, pm, pp);
      float pyp = 0.f;
#pragma unroll
      for (int t = 0; t < RK; ++t) pyp += p[t] * y[t];
      red0[wi] = wave_sum(pyp);  // the wave's lanes write the same value
      __syncthreads();
      const float quo = eta / seg_sum(red0), alpha = first ? 1.f : quo;
      float rz = 0.f;
#pragma unroll
      for (int t = 0; t < RK; ++t) r[t] -= alpha * y[t];
      if constexpr (STAIR) {
        // z = D^-1 (2 r - S w), w = D^-1 r
        float wv[RK], wm, wp;
        group_precond<RK>(R, r, wv);
        stage_w(wv);
        __syncthreads();  // staged w visible
        neighbours_w(wm, wp);
        smv(wv, wm, wp);
#pragma unroll
        for (int t = 0; t < RK; ++t) wv[t] = 2.f * r[t] - y[t];
        group_precond<RK>(R, wv, z);
      } else {
        group_precond<RK>(R, r, z);
      }
#pragma unroll
      for (int t = 0; t < RK; ++t) rz += r[t] * z[t];
      stage(z);
      red1[wi] = wave_sum(rz);
      // lambda += alpha p on the way to the barrier
      const float alpha_l = first ? 0.f : alpha;
#pragma unroll
      for (int t = 0; t < RK; ++t) lam[t] += alpha_l * p[t];
      __syncthreads();
      float zm, zp;
      neighbours(zm, zp);
      const float eta_new = seg_sum(red1);
      // taken in the last iteration too (p is not used after it)
      const float quo_b = eta_new / eta, beta = first ? 0.f : quo_b;
      eta = eta_new;
#pragma unroll
      for (int t = 0; t < RK; ++t) p[t] = fmaf(beta, p[t], z[t]);
      pm = fmaf(beta, pm, zm);
      pp = fmaf(beta, pp, zp);
      // tol < 0: exit relative to the first residual, |eta| < -tol |eta_0|
      tol_i = first && tol < 0.f ? fmaxf(-tol * fabsf(eta), FLT_MIN) : tol_i;
      ++it;
      first = false;
      conv = uniform(fabsf(eta) < tol_i);  // eta is the same in every lane
      run = !conv && it < cap;
    } while (run);
    sh.act[slot] = 0u;
  }
  // Waves that iterate no more (or have no instance) keep the others'
  // barriers until no instance of the bin iterates.  They read the act words
  // between the first two barriers, where those do not change, so all leave
  // in the same round.
  for (;;) {
    __syncthreads();
    uint32_t any = 0;
#pragma unroll
    for (int v = 0; v < MAXI; ++v) any |= sh.act[v];
    if (uniform(any == 0u)) break;
    if constexpr (STAIR) __syncthreads();
    __syncthreads();
  }

  if (!live) return;
  // (without an iteration lambda is as it was; 0 * p made NaN of an infinity)
#pragma unroll
  for (int t = 0; t < RK; ++t)
    if (it > 0 && b0 + t < N && lane_ok) lambda[(size_t)NX * (K0 + b0 + t) + i] = lam[t];
  if (lg == 0 && i == 0) {
    if (iters_out) iters_out[inst] = it;
    if (flag_out) flag_out[inst] = conv ? 0u : 1u;
    if (eta_out) eta_out[inst] = fabsf(eta);
  }
}

}  // namespace resident
}  // namespace mpc
