// One workgroup of sixteen waves runs a chain's transitions from begin to
// accept, X in its registers twice: whole rows for eta (a thread per row) and
// columns for the gradient (a thread per column of RPT DP rows).  Every wave
// keeps the chain's state, coordinate lane % DP per lane, and updates it by
// itself, so a leapfrog step has two barriers: after the residuals, and after
// the waves' partial gradients.
//
// Bound: the latency of that step, some 1500 cycles.  N = 1000, D = 10, one
// chain, twenty transitions of ten steps: 0.33 ms, against 1.89 for two
// launches per step (few_chains.h) of 3 to 4 us and what lies between them.
#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>

#include "philox.h"
#include "small_run.h"

namespace edhmc {

namespace {

constexpr int kSmallThreads = 1024, kSmallWaves = kSmallThreads / 64;
constexpr int kSmallRegs = 32;   // floats of X per thread, each way

template <int DP>
__device__ inline double coord_sum(double v) {   // over the DP coordinates, in every lane
#pragma unroll
  for (int off = 1; off < DP; off <<= 1) v += __shfl_xor(v, off, 64);
  return v;
}

template <int DP, int RPT, bool BERN>
__global__ void __launch_bounds__(kSmallThreads)
small_run_kernel(SmallArgs a) {
  constexpr int XB = RPT * DP;   // rows per thread of the gradient's products
  static_assert(XB <= kSmallRegs && 64 % DP == 0, "registers");
  __shared__ __align__(16) float rs[RPT * kSmallThreads];
  __shared__ float red[kSmallWaves][DP];
  // by the parity of the transition: with one step a transition, a wave may be
  // at the next one's sum while another still reads this one's
  __shared__ double dsum[2][kSmallWaves];
  const int c = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int d = lane % DP;
  const bool dv = d < a.D;
  const bool writes = wave == 0 && lane < DP && dv;
  LikParams lp = a.lp;
  lp.lik = BERN ? LIK_BERNOULLI : LIK_NORMAL;

  float xa[RPT][DP], xb[XB], yv[RPT];
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int64_t n = tid + (int64_t)i * kSmallThreads;
    const bool ok = n < a.N;
    yv[i] = ok ? a.y[n] : 0.0f;
#pragma unroll
    for (int k = 0; k < DP; k += 4) {   // rows are D_pad >= 64 floats, zero from D on
      f32x4_t q = {0.0f, 0.0f, 0.0f, 0.0f};
      if (ok) q = *(const f32x4_t*)(a.X + n * a.D_pad + k);
#pragma unroll
      for (int e = 0; e < 4; ++e) xa[i][k + e] = q[e];
    }
  }
  const int row0 = tid / DP * XB;
#pragma unroll
  for (int i = 0; i < XB; ++i)
    xb[i] = row0 + i < a.N ? a.X[(int64_t)(row0 + i) * a.D_pad + d] : 0.0f;

  const int64_t idx = (int64_t)c * a.D_pad + d;   // padding: z, g, loc are 0, scale is 1
  const float loc = a.ploc[d], scale = a.pscale[d], s2 = scale * scale;
  const double lscale = log((double)scale);
  float z = dv ? a.z[idx] : 0.0f, g = dv ? a.g[idx] : 0.0f, r = 0.0f, z0 = z, g0 = g, zend = z;
  double logp = a.logp[c], K0 = 0.0, ratio = 0.0;
  int n_acc = 0, n_div = 0, acc = 0;
  for (int t = 0; t < a.T; ++t) {
    const uint64_t counter = a.counter + (uint64_t)t;
    double* const ds = dsum[t & 1];
    z0 = z;
    g0 = g;
    r = 0.0f;
    if (dv) {
      if (a.r_fed) {
        r = a.r_fed[(int64_t)c * a.D + d];
      } else {
        const f32x4_t m = momentum4(a.seed, counter, (uint32_t)(d >> 2), (uint32_t)c);
        r = (d & 2) ? ((d & 1) ? m[3] : m[2]) : ((d & 1) ? m[1] : m[0]);
      }
    }
    K0 = 0.5 * coord_sum<DP>((double)r * (double)r);
    r = r + a.half * g;
    z = z + a.full * r;
    double ll = 0.0;
    for (int k = 1; k <= a.L; ++k) {
      const bool last = k == a.L;
      float eta[RPT];
#pragma unroll
      for (int i = 0; i < RPT; ++i) eta[i] = 0.0f;
#pragma unroll
      for (int q = 0; q < DP; ++q) {
        const float zq = __builtin_bit_cast(
            float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, z), q));
#pragma unroll
        for (int i = 0; i < RPT; ++i) eta[i] = fmaf(xa[i][q], zq, eta[i]);
      }
      double lls = 0.0;
#pragma unroll
      for (int i = 0; i < RPT; ++i) {
        const int n = tid + i * kSmallThreads;
        const bool ok = n < a.N;
        float dll;
        if (last) {
          double l;
          glm_both(lp, eta[i], yv[i], dll, l);
          lls += ok ? l : 0.0;
        } else {
          dll = glm_dll(lp, eta[i], yv[i]);
        }
        rs[n] = ok ? dll : 0.0f;
      }
      if (last) {
        lls = wave_sum_f64(lls);
        if (lane == 0) ds[wave] = lls;
      }
      __syncthreads();
      float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int i = 0; i < XB; i += 4) {
        const f32x4_t q = *(const f32x4_t*)(rs + row0 + i);
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] = fmaf(q[e], xb[i + e], s[e]);
      }
      float sum = (s[0] + s[1]) + (s[2] + s[3]);
#pragma unroll
      for (int off = DP; off < 64; off <<= 1) sum += __shfl_xor(sum, off, 64);
      if (lane < DP) red[wave][lane] = sum;
      __syncthreads();
      float G = 0.0f;
#pragma unroll
      for (int w = 0; w < kSmallWaves; ++w) G += red[w][d];
      g = a.lik_weight * G - (z - loc) / s2;
      r = r + a.half * g;
      if (last) {
#pragma unroll
        for (int w = 0; w < kSmallWaves; ++w) ll += ds[w];
      } else {
        r = r + a.half * g;
        z = z + a.full * r;
      }
    }
    zend = z;
    // the Metropolis test, by every wave alike
    const double tz = ((double)z - (double)loc) / (double)scale;
    const double kl = coord_sum<DP>((double)r * (double)r);
    const double plp = coord_sum<DP>(dv ? -0.5 * tz * tz - lscale - 0.5 * kLog2Pi : 0.0);
    const bool bad = __any(dv && (!isfinite(z) || !isfinite(g)));
    const double end = (double)a.lik_weight * ll + plp;
    ratio = K0 - 0.5 * kl + end - logp;
    const double u = a.u_fed ? a.u_fed[c] : accept_uniform(a.seed, counter, (uint32_t)c);
    acc = log(u) < ratio && !bad;   // NaN never accepts
    if (acc) {
      logp = end;
    } else {
      z = z0;
      g = g0;
    }
    n_acc += acc;
    n_div += bad || !(ratio == ratio);
    if (writes && a.sample_out) a.sample_out[((int64_t)t * a.C + c) * a.D + d] = z;
    if (writes && a.mom_mean) {
      const double x = z, mo = a.mom_mean[idx];
      const double mn = mo + (x - mo) / (double)(a.mom_n + t + 1);
      a.mom_mean[idx] = mn;
      a.mom_m2[idx] += (x - mo) * (x - mn);
    }
  }
  if (writes) {
    a.z[idx] = z;
    a.g[idx] = g;
    a.r[idx] = r;
    a.z0[idx] = z0;
    a.g0[idx] = g0;
    a.z_lp[idx] = zend;
  }
  __syncthreads();   // every wave has read the chain's log joint
  if (tid == 0) {
    a.logp[c] = logp;
    a.K0[c] = K0;
    if (a.accepted_out) a.accepted_out[c] = acc;
    if (a.n_accept) a.n_accept[c] += n_acc;
    if (a.ndiv) a.ndiv[c] += n_div;
    if (a.ratio_out) a.ratio_out[c] = ratio;
  }
}

int small_dp(int D) { return D <= 4 ? 4 : D <= 8 ? 8 : D <= 16 ? 16 : 32; }

}  // namespace

// The rows a thread holds, 32 floats each way: 8192 rows of up to 4 columns,
// 4096 of 8, 2048 of 16, 1024 of 32.  us per transition of ten steps, one
// or two chains, here and with few_chains.h's kernels: N = 1000, D = 10 13.4 /
// 88.6; 8192, 4 23.8 / 86.8; 4096, 8 19.9 / 90.1; 2048, 16 16.6 / 86.9; 1024,
// 32 16.8 / 82.5; 100, 3 10.7 / 82.8.  More floats per thread would spill
// (128 registers with 1024 threads).
bool small_ok(const edhmc_ctx* ctx) {
  if (!ctx->few.on || ctx->has_kinds || ctx->rec_W || ctx->D > 32) return false;
  return (ctx->N + kSmallThreads - 1) / kSmallThreads * small_dp(ctx->D) <= kSmallRegs;
}

int small_launch(edhmc_ctx* ctx, const SmallArgs& a, hipStream_t st) {
  const int rows = (int)((a.N + kSmallThreads - 1) / kSmallThreads);
  auto go = [&](auto dp, auto rpt) {
    constexpr int DP = decltype(dp)::value, RPT = decltype(rpt)::value;
    if (a.lp.lik == LIK_BERNOULLI)
      hipLaunchKernelGGL((small_run_kernel<DP, RPT, true>), dim3(a.C), dim3(kSmallThreads), 0, st, a);
    else
      hipLaunchKernelGGL((small_run_kernel<DP, RPT, false>), dim3(a.C), dim3(kSmallThreads), 0, st, a);
  };
  auto pick = [&](auto dp) {
    constexpr int DP = decltype(dp)::value, M = kSmallRegs / DP;   // most rows
    using std::integral_constant;
    if (rows <= 1) return go(dp, integral_constant<int, 1>{});
    if constexpr (M >= 2) {
      if (rows <= 2) return go(dp, integral_constant<int, 2>{});
    }
    if constexpr (M >= 4) {
      if (rows <= 4) return go(dp, integral_constant<int, 4>{});
    }
    if constexpr (M >= 8) go(dp, integral_constant<int, 8>{});
  };
  switch (small_dp(a.D)) {
    case 4: pick(std::integral_constant<int, 4>{}); break;
    case 8: pick(std::integral_constant<int, 8>{}); break;
    case 16: pick(std::integral_constant<int, 16>{}); break;
    default: pick(std::integral_constant<int, 32>{}); break;
  }
  return check_launch(ctx, "small_run");
}

}  // namespace edhmc
