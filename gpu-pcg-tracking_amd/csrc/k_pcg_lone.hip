// k_pcg_lone.hip -- PCG of one instance (N <= 128) on one workgroup, for
// gfx950: the reference-form iteration of pcg_res_body.h, laid out for the
// latency of a single solve instead of the throughput of many.
//
// Same algorithm, exit rule and arithmetic as the resident kernel (GPU-PCG
// pcg<T,14,N>, call site toplevel.cuh:143-157): block rows on 16-lane rows
// with DPP products (pcg_onchip.h), every sum in the resident kernel's order,
// so the results are bitwise its results.  What differs is how the knots are
// spread.  An iteration is a product phase, whose instructions the waves of a
// SIMD issue one after the other, and two reductions, whose latency (lane
// sums, LDS, a barrier, a division) is the same for any N.  So a short
// instance takes fewer knots per 16-lane row and more waves:
//   KR = 1 (N <= 32), 2 (N <= 64) or 4 (N <= 128) knots per row, 4 KR knots
//   per wave, up to eight waves (two per SIMD, 256 VGPRs each), which hold
//   D = S(b,b), Pinv(b,b) and the rows of S(b,b-1) and S(b+1,b) of their
//   knots in registers.
// Every wave runs every iteration (there is no other instance to wait for),
// and the loop has no branch on a value that differs between lanes.
//
// Sums.  The resident kernel sums four consecutive knots per lane ("group"),
// then a row's 16 lanes, then the four groups of 16 knots as (g0 + g1) +
// (g2 + g3), then those in order.  Here a group is spread over 4 / KR rows:
// its chain of four multiply-adds passes from row to row by a lane swap, each
// group's total goes to LDS, and after the barrier every lane reads four of
// them and the eight sums of four are added in order by DPP.
//
// One call of 173 iterations, launch included, the resident kernel (512 lanes,
// four knots per row at any N) as it was before / this one: N = 2 260 / 105
// us, N = 32 287 / 157, N = 64 328 / 201, N = 128 403 / 312.  At N = 128 a
// SIMD's two waves issue 8 knots' products (3 x 16 half-rate DPP
// multiply-adds each and 16 plain ones, about 2400 of the 4300 clocks of an
// iteration); at N <= 32 the two reductions are most of it.
#include "pcg_onchip.h"

namespace mpc {

namespace {

using namespace onchip;

constexpr int NT = 512;
constexpr int MAX_KNOTS = 128;
constexpr int MAX_GROUPS = MAX_KNOTS / 4;

struct LoneShared {
  float zb[(MAX_KNOTS + 2) * 16];   // staged vector element by knot + 1 and lane (zeros before the first and after the last)
  // group totals of the two dot products; the entry after them takes the
  // writes of the rows that end no group
  alignas(16) float red[2][MAX_GROUPS + 4];
};

// v of rows 0 and 2 in rows 1 and 3 (which = 0), or of rows 1 and 3 in rows 0
// and 2 (1)
template <int which>
__device__ __forceinline__ float swap_rows(float v) {
  const uint32_t u = __builtin_bit_cast(uint32_t, v);
  return __builtin_bit_cast(float, (uint32_t)__builtin_amdgcn_permlane16_swap(u, u, false, false)[which]);
}
// v of rows 0 and 1 in rows 2 and 3
__device__ __forceinline__ float low_to_high(float v) {
  const uint32_t u = __builtin_bit_cast(uint32_t, v);
  return __builtin_bit_cast(float, (uint32_t)__builtin_amdgcn_permlane32_swap(u, u, false, false)[0]);
}

template <int KR>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_pcg_lone(uint32_t N, const float *__restrict__ S, const float *__restrict__ Pinv, const float *__restrict__ gamma,
           float *__restrict__ lambda, uint32_t max_iter, float tol, uint32_t *__restrict__ iters_out,
           uint32_t *__restrict__ flag_out, float *__restrict__ eta_out) {
  static_assert(KR == 1 || KR == 2 || KR == 4, "knots per row");
  __shared__ LoneShared sh;
  const uint32_t tid = threadIdx.x, i = tid & 15u, q = (tid >> 4) & 3u;
  const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t d = ror_step(tid);
  for (uint32_t k = tid; k < sizeof(LoneShared) / 4; k += blockDim.x) reinterpret_cast<float *>(&sh)[k] = 0.f;
  // the row's place in the wave: knots in the order of the rows that the
  // group sums pass through, 0, 1, 3, 2 where a group takes all four
  const uint32_t place = KR == 1 ? q ^ (q >> 1) : q;
  const uint32_t b0 = 4u * KR * w + KR * place;  // first knot of the row
  const bool lane_ok = i < (uint32_t)NX;
  const uint32_t cap = pcg_cap(max_iter, N);

  Rows<KR> R;
  R.load(S, Pinv, b0, N, N, i, d);
  float lam[KR], r[KR], p[KR], y[KR], z[KR];
#pragma unroll
  for (int t = 0; t < KR; ++t) {
    const uint32_t k = b0 + (uint32_t)t;
    const bool has = lane_ok && k < N;
    lam[t] = has ? lambda[NX * k + i] : 0.f;
    r[t] = has ? gamma[NX * k + i] : 0.f;
  }
  __syncthreads();  // LDS cleared
  // the row's first and last knot staged, its neighbours' read
  float *zb0 = sh.zb + (b0 + 1u) * 16u + i;
  auto stage = [&](const float (&v)[KR]) {
    zb0[0] = v[0];
    if constexpr (KR > 1) zb0[(KR - 1) * 16] = v[KR - 1];
  };
  const float *zm_src = zb0 - 16, *zp_src = zb0 + KR * 16;
  // where the row posts its group's total: the row in which the group's chain
  // ends, the others next to the table
  const uint32_t grp = KR == 4 ? b0 >> 2 : KR == 2 ? b0 >> 2 : w;
  const bool ends = KR == 4 || (KR == 2 && (q & 1u)) || (KR == 1 && q == 2u);
  float *post_dst = &sh.red[0][ends ? grp : MAX_GROUPS];
  constexpr uint32_t RED = MAX_GROUPS + 4;
  // sum over the group's knots of u v, lane by lane, in the knots' order
  auto group_dot = [&](const float (&u)[KR], const float (&v)[KR]) {
    float s = 0.f;
#pragma unroll
    for (int t = 0; t < KR; ++t) s += u[t] * v[t];
    if constexpr (KR == 2) {
      s = swap_rows<0>(s);
#pragma unroll
      for (int t = 0; t < KR; ++t) s += u[t] * v[t];
    }
    if constexpr (KR == 1) {
      s = swap_rows<0>(s);  // row 0 -> 1
      s += u[0] * v[0];
      s = low_to_high(s);   // row 1 -> 3
      s += u[0] * v[0];
      s = swap_rows<1>(s);  // row 3 -> 2
      s += u[0] * v[0];
    }
    return s;
  };
  auto post = [&](int k, float s) { post_dst[k * RED] = row_total(s); };
  // ((g0 + g1) + (g2 + g3)) of every 16 knots, then those in order
  auto total = [&](int k) {
    const float4 g = *reinterpret_cast<const float4 *>(&sh.red[k][4u * (i & 7u)]);
    const float v = (g.x + g.y) + (g.z + g.w);
    float s = v;
    if constexpr (KR == 1)
      asm("s_nop 1\n"
          "v_mov_b32_dpp %0, %1 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
          "v_add_f32_dpp %0, %1, %0 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
          : "=&v"(s)
          : "v"(v));
    else if constexpr (KR == 2)
      asm("s_nop 1\n"
          "v_mov_b32_dpp %0, %1 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
          "v_add_f32_dpp %0, %1, %0 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
          "v_add_f32_dpp %0, %1, %0 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
          "v_add_f32_dpp %0, %1, %0 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
          : "=&v"(s)
          : "v"(v));
    else
      asm("s_nop 1\n"
          "v_mov_b32_dpp %0, %1 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
          "v_add_f32_dpp %0, %1, %0 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
          "v_add_f32_dpp %0, %1, %0 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
          "v_add_f32_dpp %0, %1, %0 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
          "v_add_f32_dpp %0, %1, %0 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
          "v_add_f32_dpp %0, %1, %0 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
          "v_add_f32_dpp %0, %1, %0 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
          "v_add_f32_dpp %0, %1, %0 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
          : "=&v"(s)
          : "v"(v));
    return s;
  };
  stage(lam);
  __syncthreads();
  float pm = *zm_src, pp = *zp_src;

  // The first pass is the prologue, through the same code: p = lambda,
  // r = gamma - S lambda (alpha = 1, lambda kept), z = Pinv r, then p = z
  // (beta = 0) and eta = r.z; the others are the iterations.
#pragma unroll
  for (int t = 0; t < KR; ++t) p[t] = lam[t];
  uint32_t it = ~0u;  // the first pass is not counted
  float eta = 0.f;
  bool first = true, conv, run;
  do {
    group_smv<KR>(R, p, pm, pp, y);
    post(0, group_dot(p, y));
    __syncthreads();
    const float quo = eta / total(0), alpha = first ? 1.f : quo;
    // (knot by knot: all updates first cost 1 % of a solve)
#pragma unroll
    for (int t = 0; t < KR; ++t) {
      r[t] -= alpha * y[t];
      z[t] = row_precond(R.P[t], r[t]);
    }
    stage(z);
    post(1, group_dot(r, z));
    __syncthreads();
    const float zm = *zm_src, zp = *zp_src, eta_new = total(1);
    const float alpha_l = first ? 0.f : alpha;
#pragma unroll
    for (int t = 0; t < KR; ++t) lam[t] += alpha_l * p[t];
    // taken in the last iteration too (p is not used after it)
    const float quo_b = eta_new / eta, beta = first ? 0.f : quo_b;
    eta = eta_new;
#pragma unroll
    for (int t = 0; t < KR; ++t) p[t] = fmaf(beta, p[t], z[t]);
    pm = fmaf(beta, pm, zm);
    pp = fmaf(beta, pp, zp);
    ++it;
    first = false;
    conv = uniform(fabsf(eta) < tol);  // eta is the same in every lane
    run = !conv && it < cap;
  } while (run);

  // (without an iteration lambda is as it was; 0 * p made NaN of an infinity)
  if (it > 0) {
#pragma unroll
    for (int t = 0; t < KR; ++t)
      if (b0 + t < N && lane_ok) lambda[NX * (b0 + t) + i] = lam[t];
  }
  if (tid == 0) {
    if (iters_out) *iters_out = it;
    if (flag_out) *flag_out = conv ? 0u : 1u;
    if (eta_out) *eta_out = fabsf(eta);
  }
}

template <int KR>
hipError_t launch_knots(uint32_t N, const float *S, const float *Pinv, const float *gamma, float *lambda,
                        uint32_t max_iter, float tol, uint32_t *iters, uint32_t *flag, float *eta, hipStream_t st) {
  const uint32_t waves = (N + 4u * KR - 1u) / (4u * KR);
  hipLaunchKernelGGL((k_pcg_lone<KR>), dim3(1), dim3(64u * waves), 0, st, N, S, Pinv, gamma, lambda, max_iter, tol,
                     iters, flag, eta);
  return hipGetLastError();
}

}  // namespace

uint32_t pcg_lone_max_knots() { return (uint32_t)MAX_KNOTS; }

// as few knots per row as eight waves allow
hipError_t launch_pcg_lone(uint32_t N, const float *S, const float *Pinv, const float *gamma, float *lambda,
                           uint32_t max_iter, float tol, uint32_t *iters, uint32_t *flag, float *eta, hipStream_t st) {
  if (N < 1 || N > (uint32_t)MAX_KNOTS) return hipErrorInvalidValue;
  if (N <= 32u) return launch_knots<1>(N, S, Pinv, gamma, lambda, max_iter, tol, iters, flag, eta, st);
  if (N <= 64u) return launch_knots<2>(N, S, Pinv, gamma, lambda, max_iter, tol, iters, flag, eta, st);
  return launch_knots<4>(N, S, Pinv, gamma, lambda, max_iter, tol, iters, flag, eta, st);
}

}  // namespace mpc
