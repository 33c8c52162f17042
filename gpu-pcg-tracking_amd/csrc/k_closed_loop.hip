// k_closed_loop.hip -- device side of the closed-loop tracking harness
// (gfx950): plant simulation, state noise, tracking error and the receding-
// horizon shift of one control step, in one single-workgroup kernel, so a
// control step is the batched SQP launch sequence plus this kernel and
// needs no host round trip (and can be captured in a HIP graph).
//
// The plant is a serial chain, and a wave alone on its SIMD issues one
// instruction in four clocks, so its time is the number of instructions of a
// substep.  Two waves share them: positions step by the velocities alone, so
// one wave is a substep ahead with sines, columns of M and factor (about 700)
// while the other takes bias forces, solve and step (about 700).  The other
// waves read the plan's shifted parts and draw the noise meanwhile.  A control
// step of 50 substeps at N = 128: 150 us in one wave that did it all in turn
// (1400 instructions a substep, the plan in 70 trips to memory), 76 us so.
//
// Reference: track() (toplevel.cuh:505-775) with simple_simulate /
// simple_integrator_kernel (integrator.cuh:283-398) and just_shift
// (integrator.cuh:283-289).  Control step s (one knot: the plan shifts by
// one knot per step, so substeps * sim_dt is the knot interval):
//   1. the SQP (separate launches) has solved the plan xu from x_s;
//   2. plant: `substeps` explicit Euler steps of sim_dt (the reference's
//      integrator type 0: q += h qd, qd += h qdd(q, qd, u)) under the
//      plan's first control u_0 (zero-order hold);
//   3. state noise: x += sigma n, n ~ N(0, I) from splitmix64 + Box-Muller
//      (pair i of step s seeded with seed ^ 0xD1B54A32D192ED03 (8 s + i + 1));
//   4. error: ee(q_{s+1}) - ref_{s+1} (xyz), Euclidean and L1 norms;
//   5. shift: x_k <- x_{k+1}, u_k <- u_{k+1}, lambda_k <- lambda_{k+1};
//      the new tail (u_{N-2}, x_{N-1}) from the precomputed trajectory
//      (its u_{s+N-1}, x_{s+N}; the reference fills the tail from its
//      precomputed trajectory too, toplevel.cuh:680-690) or, without one,
//      u_{N-2} <- 0 and x_{N-1} kept; reference window <- path[s+1 .. s+N];
//      x_0 <- the plant state.
// Differences from the reference: the reference's plant runs the previous
// plan during the solve time (CONST_UPDATE_FREQ, SIMULATION_PERIOD) and
// shifts once per knot interval; here every control step is one knot
// interval and the new plan's u_0 is applied.  Noise: the reference's
// noise.cuh is disabled and faulty; this is the harness's own definition.
#include "common.h"
#include "model.h"

namespace mpc {

namespace {

constexpr int NT = 64;    // k_cl_init: one wave
constexpr int SNT = 512;  // k_cl_step: the plant's two waves and six that shift the plan
constexpr int SHIFT_NT = SNT - 128, SHIFT_PER = 16;

struct alignas(16) ClLds {
  float fac[2][40];          // by substep: the factor of M by columns (28), its refined reciprocals (7), 1 if divisions need scaling
  float sn[2][8], cs[2][8];  // by substep
  float x[2][16];            // by substep
  float M[49];
  float u[8];
  float noise[16];
};

// no multiply-add across this point
__device__ __forceinline__ void keep(float &v) { asm("" : "+v"(v)); }

// rnea at qd = 0 and qdd = the lane's unit vector, to the bit: the terms in
// the velocities are exact zeros, and from link 2 up they are left out (the
// sums that one of them enters in rnea, v x S qd in the accelerations and
// v x* I v in the forces, kept from becoming part of a multiply-add); the
// first two links, where the model's constants fold most of it, run as they
// stand there, with zeros that the compiler does not know.
__device__ __forceinline__ void rnea_unit(const float *s, const float *c, const float *qdd, float *tau) {
  float f[NQ][6], vp[6] = {0, 0, 0, 0, 0, 0}, ap[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    float a[6];
    if (i < 2) {
      float v[6], qd = 0.f;
      keep(qd);
      X_mv(i, s[i], c[i], vp, v);
      X_mv(i, s[i], c[i], ap, a);
      v[2] += qd;
      a[2] += qdd[i];
      const float sq[6] = {0, 0, qd, 0, 0, 0};
      float t[6], Ia[6], Iv[6], cf[6];
      crm(v, sq, t);
#pragma unroll
      for (int k = 0; k < 6; ++k) a[k] += t[k];
      inertia_mv(i, a, Ia);
      inertia_mv(i, v, Iv);
      crf(v, Iv, cf);
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        f[i][k] = Ia[k] + cf[k];
        vp[k] = v[k];
      }
    } else {
      X_mv(i, s[i], c[i], ap, a);
      a[2] += qdd[i];
      keep(a[0]);
      keep(a[1]);
      keep(a[3]);
      keep(a[4]);
      inertia_mv(i, a, f[i]);
#pragma unroll
      for (int k = 0; k < 6; ++k) keep(f[i][k]);
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) ap[k] = a[k];
  }
#pragma unroll
  for (int i = NQ - 1; i >= 0; --i) {
    tau[i] = f[i][2];
    if (i > 0) {
      float t[6];
      XT_fv(i, s[i], c[i], f[i], t);
#pragma unroll
      for (int k = 0; k < 6; ++k) f[i - 1][k] += t[k];
    }
  }
}

// 2^-46 .. 2^46: quotients of such values take no scaling
constexpr float DIV_MIN = 0x1p-46f, DIV_MAX = 0x1p46f;

// cholesky7, and the refined reciprocals r of the diagonal; the inverses by the
// division's own sequence without its scaling and fix-up, so the same as long
// as the diagonal lies in DIV_MIN .. DIV_MAX (returned)
__device__ __forceinline__ bool cholesky7_quick(const float *M, float *L, float *r) {
  float lo = DIV_MIN, hi = DIV_MAX;
#pragma unroll
  for (int j = 0; j < NQ; ++j) {
    float d = M[j + 7 * j];
#pragma unroll
    for (int k = 0; k < j; ++k) d -= L[j + 7 * k] * L[j + 7 * k];
    d = sqrtf(d);
    lo = fminf(lo, d);
    hi = fmaxf(hi, d);
    L[j + 7 * j] = d;
    const float r0 = __builtin_amdgcn_rcpf(d);
    r[j] = fmaf(fmaf(-d, r0, 1.f), r0, r0);
    float inv = fmaf(fmaf(-d, r[j], 1.f), r[j], r[j]);
    inv = fmaf(fmaf(-d, inv, 1.f), r[j], inv);
#pragma unroll
    for (int i = j + 1; i < NQ; ++i) {
      float s = M[i + 7 * j];
#pragma unroll
      for (int k = 0; k < j; ++k) s -= L[i + 7 * k] * L[j + 7 * k];
      L[i + 7 * j] = s * inv;
    }
  }
  return lo == DIV_MIN && hi == DIV_MAX;
}

// x = L^-T L^-1 b as chol_solve7, with r[i] the refined reciprocal of L(i, i):
// the rest of the division's own sequence without its scaling and fix-up, so
// the same quotients as long as every numerator lies in DIV_MIN .. DIV_MAX
// (returned).
__device__ __forceinline__ bool chol_solve7_quick(const float *L, const float *r, const float *b, float *x) {
  float y[NQ], lo = DIV_MIN, hi = DIV_MAX;
  auto quotient = [&](float s, int i) {
    lo = fminf(lo, fabsf(s));
    hi = fmaxf(hi, fabsf(s));
    const float d = L[i + 7 * i];
    float q = s * r[i];
    q = fmaf(fmaf(-d, q, s), r[i], q);
    return fmaf(fmaf(-d, q, s), r[i], q);
  };
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    float s = b[i];
#pragma unroll
    for (int k = 0; k < i; ++k) s -= L[i + 7 * k] * y[k];
    y[i] = quotient(s, i);
  }
#pragma unroll
  for (int i = NQ - 1; i >= 0; --i) {
    float s = y[i];
#pragma unroll
    for (int k = i + 1; k < NQ; ++k) s -= L[k + 7 * i] * x[k];
    x[i] = quotient(s, i);
  }
  return lo == DIV_MIN && hi == DIV_MAX;
}

__device__ __forceinline__ uint64_t sm64(uint64_t &s) {
  uint64_t z = (s += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// pair i (< 7) of the step's 14 standard normals
__device__ __forceinline__ void noise_pair(uint64_t seed, uint32_t step, uint32_t i, float &a, float &b) {
  uint64_t s = seed ^ (0xD1B54A32D192ED03ull * (8ull * step + i + 1ull));
  const double u1 = (double)((sm64(s) >> 11) + 1ull) * 0x1.0p-53;  // (0, 1]
  const double u2 = (double)(sm64(s) >> 11) * 0x1.0p-53;           // [0, 1)
  const double r = sqrt(-2.0 * log(u1));
  const double t = 6.283185307179586 * u2;
  a = (float)(r * cos(t));
  b = (float)(r * sin(t));
}

__global__ void __launch_bounds__(NT) k_cl_init(uint32_t N, const float *__restrict__ x0,
                                                const float *__restrict__ path, float *__restrict__ win,
                                                float *__restrict__ xu, float *__restrict__ xp,
                                                uint32_t *__restrict__ ctr, float *__restrict__ states,
                                                float *__restrict__ rho, float rho0) {
  const uint32_t t = threadIdx.x;
  if (t < NX) {
    const float v = x0[t];
    xp[t] = v;
    xu[t] = v;
    states[t] = v;
  }
  for (uint32_t j = t; j < 6 * N; j += NT) win[j] = path[j];
  if (t == 0) {
    ctr[0] = 0;
    rho[0] = rho0;
  }
}

// One chunk of a shift in place, dst[j] <- dst[j + by] for j0 <= j < n, on
// the lanes u of the shift waves: read() ahead of a workgroup barrier,
// write() behind it.  (A chunk's reads reach `by` elements into the next one,
// which is written later.)
struct ShiftChunk {
  float v[SHIFT_PER];
  __device__ __forceinline__ void read(const float *src, uint32_t by, uint32_t j0, uint32_t n, uint32_t u) {
#pragma unroll
    for (int k = 0; k < SHIFT_PER; ++k) {
      const uint32_t j = j0 + u + (uint32_t)(k * SHIFT_NT);
      v[k] = j < n ? src[j + by] : 0.f;
    }
  }
  __device__ __forceinline__ void write(float *dst, uint32_t j0, uint32_t n, uint32_t u) const {
#pragma unroll
    for (int k = 0; k < SHIFT_PER; ++k) {
      const uint32_t j = j0 + u + (uint32_t)(k * SHIFT_NT);
      if (j < n) dst[j] = v[k];
    }
  }
};

__global__ void __launch_bounds__(SNT) k_cl_step(ClStep p, const float *__restrict__ path,
                                                 const float *__restrict__ traj, float *__restrict__ win,
                                                 float *__restrict__ xu, float *__restrict__ lam,
                                                 float *__restrict__ xp, uint32_t *__restrict__ ctr,
                                                 float *__restrict__ states, float *__restrict__ err,
                                                 const uint32_t *__restrict__ pcg_now,
                                                 uint32_t *__restrict__ pcg_log) {
  __shared__ ClLds L;
  const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t t = threadIdx.x & 63u;
  const bool shifts = w >= 2u;
  const uint32_t u = threadIdx.x - 128u;  // lane of the shift waves
  const uint32_t step = ctr[0];
  const uint32_t N = p.N;
  if (w == 0) {
    if (t < NX) L.x[0][t] = xp[t];
    if (t < NU) L.u[t] = xu[NX + t];
  }
  // 5. shift: the first chunks are read while the plant runs
  const uint32_t nsh = NXU * N - NU - NXU, nl = NX * (N - 1);
  ShiftChunk cx, cl;
  if (shifts) {
    cx.read(xu, NXU, 0, nsh, u);
    cl.read(lam, NX, 0, nl, u);
    if (u < NQ && p.sigma > 0.f) noise_pair(p.seed, step, u, L.noise[2 * u], L.noise[2 * u + 1]);
  }
  __syncthreads();
  // 2. plant: explicit Euler substeps under u_0.  The positions of the next
  // substep need no acceleration, so wave 0 is one ahead: its sines, columns
  // of M and factor, while wave 1 takes this substep's bias forces, solves
  // and steps.
  auto mass_factor = [&](float q, uint32_t buf) {  // q: joint t's position
    if (t < NQ) {
      float s, c;
      sincosf(q, &s, &c);
      L.sn[buf][t] = s;
      L.cs[buf][t] = c;
    }
    wave_sync();
    float s[NQ], c[NQ], qdd[NQ], tau[NQ], Lc[49], rd[NQ];
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      s[i] = L.sn[buf][i];
      c[i] = L.cs[buf][i];
      qdd[i] = i == (int)t ? 1.f : 0.f;
    }
    rnea_unit(s, c, qdd, tau);  // lanes 0..6: column t of M = RNEA(q, 0, e_t)
    if (t < NQ) {
#pragma unroll
      for (int r = 0; r < NQ; ++r) L.M[r + 7 * t] = tau[r];
    }
    wave_sync();
    const bool quick = cholesky7_quick(L.M, Lc, rd);
    if (!quick) cholesky7(L.M, Lc);
    float *o = L.fac[buf];  // (every lane the same)
    int n = 0;
#pragma unroll
    for (int j = 0; j < NQ; ++j)
#pragma unroll
      for (int i = j; i < NQ; ++i) o[n++] = Lc[i + 7 * j];
#pragma unroll
    for (int j = 0; j < NQ; ++j) o[28 + j] = rd[j];
    o[35] = quick ? 0.f : 1.f;
  };
  for (uint32_t stage = 0; stage <= p.substeps; ++stage) {
    // stage k: M of substep k, the step of substep k - 1
    const uint32_t nxt = stage & 1u, now = nxt ^ 1u;
    if (w == 0 && stage < p.substeps) {
      const float dt = stage > 0 ? p.sim_dt : 0.f;
      const uint32_t from = stage > 0 ? now : 0u;
      mass_factor(t < NQ ? L.x[from][t] + dt * L.x[from][NQ + t] : 0.f, nxt);
    } else if (w == 1 && stage > 0) {
      // bias RNEA(q, qd, 0); qdd = 0 not known to the compiler, which would
      // form other multiply-adds without the additions
      float s[NQ], c[NQ], qd[NQ], zero[NQ], bias[NQ], fac[40], Lc[49], rhs[NQ], qdd[NQ];
#pragma unroll
      for (int i = 0; i < NQ; ++i) {
        s[i] = L.sn[now][i];
        c[i] = L.cs[now][i];
        qd[i] = L.x[now][NQ + i];
        zero[i] = 0.f;
        keep(zero[i]);
      }
#pragma unroll
      for (int k = 0; k < 36; ++k) fac[k] = L.fac[now][k];
      rnea<false>(s, c, qd, zero, bias, nullptr, nullptr, nullptr, nullptr, nullptr);
      int n = 0;
#pragma unroll
      for (int j = 0; j < NQ; ++j)
#pragma unroll
        for (int i = j; i < NQ; ++i) Lc[i + 7 * j] = fac[n++];
#pragma unroll
      for (int i = 0; i < NQ; ++i) rhs[i] = L.u[i] - bias[i];
      if (!chol_solve7_quick(Lc, fac + 28, rhs, qdd) || fac[35] != 0.f) chol_solve7(Lc, rhs, qdd);
      float a = qdd[0];
#pragma unroll
      for (int i = 1; i < NQ; ++i) a = (int)t == i ? qdd[i] : a;
      if (t < NQ) {
        const float q = L.x[now][t], v = L.x[now][NQ + t];
        L.x[nxt][t] = q + p.sim_dt * v;
        L.x[nxt][NQ + t] = v + p.sim_dt * a;
      }
    }
    __syncthreads();
  }
  float *x = L.x[p.substeps & 1u];
  // 3. noise
  if (w == 0 && t < NQ && p.sigma > 0.f) {
    x[2 * t] += p.sigma * L.noise[2 * t];
    x[2 * t + 1] += p.sigma * L.noise[2 * t + 1];
  }
  __syncthreads();
  if (w == 0) {
    if (t < NX) {
      xp[t] = x[t];
      states[(size_t)NX * (step + 1) + t] = x[t];
    }
    if (pcg_log && t < p.sqp_iters) pcg_log[(size_t)p.sqp_iters * step + t] = pcg_now[t];
  } else if (w == 1) {
    // 4. tracking error against the reference point of the new time
    if (t < NQ) {
      float s, c;
      sincosf(x[t], &s, &c);
      L.sn[1][t] = s;
      L.cs[1][t] = c;
    }
    wave_sync();
    if (t == 0) {
      float s[NQ], c[NQ], ee[3];
#pragma unroll
      for (int i = 0; i < NQ; ++i) {
        s[i] = L.sn[1][i];
        c[i] = L.cs[1][i];
      }
      fk_pos(s, c, ee);
      const float *r = path + (size_t)6 * (step + 1);
      const float e0 = ee[0] - r[0], e1 = ee[1] - r[1], e2 = ee[2] - r[2];
      err[2 * step] = sqrtf(e0 * e0 + e1 * e1 + e2 * e2);
      err[2 * step + 1] = fabsf(e0) + fabsf(e1) + fabsf(e2);
    }
  }
  // 5. shift, the first chunks from registers
  if (shifts) {
    cx.write(xu, 0, nsh, u);
    cl.write(lam, 0, nl, u);
    for (uint32_t j = u; j < 6 * N; j += SHIFT_NT) win[j] = path[(size_t)6 * (step + 1) + j];
  }
  constexpr uint32_t CHUNK = SHIFT_NT * SHIFT_PER;
  const uint32_t n_shift = nsh > nl ? nsh : nl;
  for (uint32_t j0 = CHUNK; j0 < n_shift; j0 += CHUNK) {
    if (shifts) {
      cx.read(xu, NXU, j0, nsh, u);
      cl.read(lam, NX, j0, nl, u);
    }
    __syncthreads();
    if (shifts) {
      cx.write(xu, j0, nsh, u);
      cl.write(lam, j0, nl, u);
    }
  }
  __syncthreads();
  if (w == 0) {
    if (traj) {
      if (t < NXU) xu[NXU * (N - 2) + NX + t] = traj[(size_t)NXU * (step + N - 1) + NX + t];
    } else if (t < NU) {
      xu[NXU * (N - 2) + NX + t] = 0.f;
    }
    if (t < NX) xu[t] = x[t];
    if (t == 0) ctr[0] = step + 1;
  }
}

}  // namespace

hipError_t launch_cl_init(uint32_t N, const float *x0, const float *path, float *win, float *xu, float *xp,
                          uint32_t *ctr, float *states, float *rho, float rho0, hipStream_t st) {
  hipLaunchKernelGGL(k_cl_init, dim3(1), dim3(NT), 0, st, N, x0, path, win, xu, xp, ctr, states, rho, rho0);
  return hipGetLastError();
}

hipError_t launch_cl_step(const ClStep &p, const float *path, const float *traj, float *win, float *xu, float *lam,
                          float *xp, uint32_t *ctr, float *states, float *err, const uint32_t *pcg_now,
                          uint32_t *pcg_log, hipStream_t st) {
  if (p.N < 2 || p.sqp_iters > NT) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_cl_step, dim3(1), dim3(SNT), 0, st, p, path, traj, win, xu, lam, xp, ctr, states, err,
                     pcg_now, pcg_log);
  return hipGetLastError();
}

}  // namespace mpc
