// Readout of sample stores on MI355X: column moments (Empirical.mean /
// variance, edward/models/empirical.py:87-96) and the multi-chain
// autocovariances behind the effective sample size (no reference
// counterpart).  All sums in FP64, in a fixed order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"
#include "ctx.h"

using namespace edhmc;

namespace edhmc {
bool autocov_fft_ok(int64_t T, int n_lags);
int autocov_fft_block(int64_t T, int D);
int autocov_fft(edhmc_ctx* ctx, const float* s, int64_t T, int C, int D, int d0, int db, int n_lags,
                double* mean, int64_t ldm, double* acov, int64_t ld, hipStream_t st);
int ess_launch(edhmc_ctx* ctx, const double* acov, const double* mean, int64_t T, int C, int D,
               bool between, double* ess, hipStream_t st);
}  // namespace edhmc

namespace {

// ---------------------------------------------------------------------------
// Column moments of x [T, K] over rows t0 .. T-1: mean and population variance
// (var == nullptr: the mean alone).
//
// A workgroup of NT threads takes CW adjacent columns and deals the rows
// round-robin to NT / CW groups of threads.  A thread takes kMomRows rows at
// a time, the next ones loading meanwhile, and merges their sum and squared
// deviations from their own mean into its running ones (Chan, Golub, LeVeque
// 1979), so x is read once whatever T is, 1 KB of a row at a time in a wide
// store.  Bound by the read of x; T = 1000, K = 262,144 (1.05 GB): 210
// us, 5.0 TB/s (64 columns at a time, the rows in registers: 616).
// ---------------------------------------------------------------------------
constexpr int kMomRows = 16;

struct Moments {
  double n, sum, dev;   // rows, their sum, squared deviations from their mean
};

__device__ inline Moments merge(const Moments& a, const Moments& b) {
  if (b.n == 0.0) return a;
  if (a.n == 0.0) return b;
  const double n = a.n + b.n, d = b.sum / b.n - a.sum / a.n;
  return {n, a.sum + b.sum, a.dev + b.dev + d * d * (a.n * b.n / n)};
}

template <typename P, int NT>
__global__ void __launch_bounds__(NT)
moments_kernel(const P* __restrict__ x, int64_t T, int64_t K, int64_t t0, int cw,
               double* __restrict__ mean, double* __restrict__ var) {
  __shared__ Moments sm[NT];
  const int tid = threadIdx.x, groups = NT / cw;
  const int64_t k = (int64_t)blockIdx.x * cw + (tid & (cw - 1));
  const int g = tid / cw;
  const int64_t n = T - t0;
  const int64_t mine = g < n ? (n - g + groups - 1) / groups : 0;   // rows g, g + groups, ...
  const P* p = x + (t0 + g) * K + min(k, K - 1);
  const int64_t step = (int64_t)groups * K;
  P v[kMomRows];
  auto load = [&](int64_t i0) {
#pragma unroll
    for (int i = 0; i < kMomRows; ++i) v[i] = i0 + i < mine ? p[(i0 + i) * step] : (P)0;
  };
  Moments a = {0.0, 0.0, 0.0};
  load(0);
  for (int64_t i0 = 0; i0 < mine; i0 += kMomRows) {
    P w[kMomRows];
#pragma unroll
    for (int i = 0; i < kMomRows; ++i) w[i] = v[i];
    if (i0 + kMomRows < mine) load(i0 + kMomRows);
    const int cnt = (int)min((int64_t)kMomRows, mine - i0);
    Moments b = {(double)cnt, 0.0, 0.0};
#pragma unroll
    for (int i = 0; i < kMomRows; ++i) b.sum += (double)w[i];   // zeros from cnt on
    const double m = b.sum / b.n;
#pragma unroll
    for (int i = 0; i < kMomRows; ++i) {
      const double d = (double)w[i] - m;
      b.dev += i < cnt ? d * d : 0.0;
    }
    a = merge(a, b);
  }
  sm[tid] = a;
  __syncthreads();
  for (int w = NT / 2; w >= cw; w >>= 1) {
    if (tid < w) sm[tid] = merge(sm[tid], sm[tid + w]);
    __syncthreads();
  }
  if (g != 0 || k >= K) return;
  a = sm[tid];
  mean[k] = a.sum / a.n;
  if (var) var[k] = a.dev / a.n;
}

template <typename P>
int launch_moments(edhmc_ctx* ctx, const P* x, int64_t T, int64_t K, int64_t t0, double* mean,
                   double* var, hipStream_t st) {
  // columns per workgroup: 256 where that leaves a thousand workgroups, down
  // to 64, fewer for a narrow store; 1024 threads (rows in more groups) where
  // there are few workgroups, but not for rows that 256 threads hold at once
  // (64 x 51,200: 19.3 us with 1024, 6.5 with 256; 6.5 for 64 x 6000 either way)
  int cw = 4;
  while (cw < 64 && cw < K) cw *= 2;
  while (cw >= 64 && cw < 256 && K / (2 * cw) >= 1024) cw *= 2;
  const int64_t blocks = (K + cw - 1) / cw;
  if (blocks > 2147483647LL) return set_err(ctx, EDHMC_EUNSUPPORTED, "too many columns");
  const dim3 grid((unsigned)blocks);
  if (blocks >= 1024 || (T - t0) * cw <= 256 * kMomRows)
    hipLaunchKernelGGL((moments_kernel<P, 256>), grid, dim3(256), 0, st, x, T, K, t0, cw, mean, var);
  else
    hipLaunchKernelGGL((moments_kernel<P, 1024>), grid, dim3(1024), 0, st, x, T, K, t0, cw, mean, var);
  return check_launch(ctx, "moments");
}

// ---------------------------------------------------------------------------
// Autocovariances at lags lag0 .. lag0 + n_lags - 1 of the chains of a store
// s [T, C, D], summed over the chains: per series sum_t a_t a_{t + lag} with
// a = x - chain mean, in FP64.
//
// A lane owns one column v of P = D m adjacent ones (m chains side by side,
// so that narrow stores fill a wave) and LAGS lags, whose sums stay in
// registers over all the chains of its group.  With 32 lags, per step of 8
// draws it loads 8 new a_t and 8 new a_{t + lag} (the window of 40 rotates
// through five register arrays) and issues 256 FP64 FMAs; the waves of a
// workgroup take adjacent lag blocks of the same columns, and the workgroups
// of one column strip and chain group run on one XCD, so the store is read
// from its L2.  Bound by the FP64 FMAs (n_lags (T - lag) C D of them) and the
// wait for the loads.  T = 1000, C = 1024, D = 256, all 1000 lags in five
// windows: 14.8 ms, against 105 ms for a thread per series with one atomic per
// series and lag.  It takes windows that do not begin at lag 0, at most 32
// lags, and more than 2048 draws (acov_fft.hip the others), and whatever has
// to do without scratch: then one group, chains one after the other, its sums
// straight in the output.  OWN_MEAN: it makes the chain means itself.
// ---------------------------------------------------------------------------
constexpr int kAcStep = 8, kAcWaves = 4;
constexpr int64_t kAcPartBytes = 128 << 20;     // partial sums

struct AcovArgs {
  const float* s;
  int64_t T;
  int C, D, m, P;          // chains, columns, chains side by side, P = D m
  int lag0, n_lags;
  int blocks, groups;      // chain blocks of m chains, groups of them
  int strips, lag_wgs;     // 64-column strips of P, workgroups along the lags
  double* mean;            // [C][D] (OWN_MEAN: written, or null)
  double* part;            // [groups][n_lags][P]
};

template <int LAGS, bool OWN_MEAN>
__global__ void __launch_bounds__(64 * kAcWaves) __attribute__((amdgpu_waves_per_eu(LAGS > 8 ? 1 : 4, LAGS > 8 ? 2 : 8)))
autocov_kernel(AcovArgs a) {
  constexpr int WIN = LAGS / kAcStep + 1;   // window of WIN kAcStep values
  // units (strip, chain group) dealt to the XCDs, all lags of a unit on one
  const int units = a.strips * a.groups;
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int unit = xcd + 8 * (local / a.lag_wgs);
  if (unit >= units) return;
  const int strip = unit % a.strips, grp = unit / a.strips;
  const int lane = threadIdx.x & 63;
  // uniform over the wave: times and row addresses stay in scalar registers
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lb = (local % a.lag_wgs) * (blockDim.x >> 6) + wave;   // lag block of this wave
  if (lb * LAGS >= a.n_lags) return;
  const int64_t l0 = (int64_t)a.lag0 + (int64_t)lb * LAGS;
  const int v = strip * 64 + lane;
  const int j = v / a.D, d = v - j * a.D;
  const int64_t stride = (int64_t)a.C * a.D;
  const int64_t T = a.T;

  double acc[LAGS];
#pragma unroll
  for (int l = 0; l < LAGS; ++l) acc[l] = 0.0;
  const int per = (a.blocks + a.groups - 1) / a.groups;
  const int k1 = min(a.blocks, (grp + 1) * per);
  for (int k = grp * per; k < k1; ++k) {
    const int c = k * a.m + j;
    if (v >= a.P || c >= a.C) continue;
    const float* p = a.s + (int64_t)k * a.m * a.D;   // row of draw 0; the lane reads column v
    auto x_at = [&](int64_t t) -> float { return (p + min(t, T - 1) * stride)[(uint32_t)v]; };
    double mean;
    if constexpr (OWN_MEAN) {
      mean = 0.0;
#pragma unroll 16
      for (int64_t t = 0; t < T; ++t) mean += (double)x_at(t);
      mean /= (double)T;
      if (lb == 0 && a.mean) a.mean[(int64_t)c * a.D + d] = mean;
    } else {
      mean = a.mean[(int64_t)c * a.D + d];
    }
    double w[WIN][kAcStep];
    // a_t at times past the last draw read as 0
#pragma unroll
    for (int q = 0; q < WIN - 1; ++q)
#pragma unroll
      for (int i = 0; i < kAcStep; ++i) {
        const int64_t t = l0 + q * kAcStep + i;
        w[q][i] = t < T ? (double)x_at(t) - mean : 0.0;
      }
    const int64_t t_end = T - l0;   // draws with a partner at lag l0
    // raw values of the coming step, loaded one step ahead (past the end: the
    // last draw again, masked or multiplied by 0)
    float ra[kAcStep], rw[kAcStep];
    auto fetch = [&](int64_t t) {
#pragma unroll
      for (int i = 0; i < kAcStep; ++i) {
        ra[i] = x_at(t + i);
        rw[i] = x_at(t + l0 + LAGS + i);
      }
    };
    fetch(0);
    // step at draws t .. t + 7, the window's oldest array being w[r]
    auto step = [&](int64_t t, auto rc) {
      constexpr int r = decltype(rc)::value;
      double x[kAcStep];
      const int64_t tw = t + l0 + LAGS;
#pragma unroll
      for (int i = 0; i < kAcStep; ++i) {
        x[i] = (double)ra[i] - mean;
        w[(r + WIN - 1) % WIN][i] = tw + i < T ? (double)rw[i] - mean : 0.0;
      }
      if (t + kAcStep < t_end) fetch(t + kAcStep);
#pragma unroll
      for (int i = 0; i < kAcStep; ++i)
#pragma unroll
        for (int l = 0; l < LAGS; ++l) {
          const int q = i + l;
          acc[l] = fma(x[i], w[(r + q / kAcStep) % WIN][q % kAcStep], acc[l]);
        }
    };
    using std::integral_constant;
    static_assert(WIN == 2 || WIN == 5, "steps of a turn of the window");
    for (int64_t t = 0; t < t_end; t += WIN * kAcStep) {
      step(t, integral_constant<int, 0>{});
      if (t + kAcStep < t_end) step(t + kAcStep, integral_constant<int, 1>{});
      if constexpr (WIN == 5) {
        if (t + 2 * kAcStep < t_end) step(t + 2 * kAcStep, integral_constant<int, 2>{});
        if (t + 3 * kAcStep < t_end) step(t + 3 * kAcStep, integral_constant<int, 3>{});
        if (t + 4 * kAcStep < t_end) step(t + 4 * kAcStep, integral_constant<int, 4>{});
      }
    }
  }
  if (v >= a.P) return;
#pragma unroll
  for (int l = 0; l < LAGS; ++l)
    if (lb * LAGS + l < a.n_lags)
      a.part[((int64_t)grp * a.n_lags + lb * LAGS + l) * a.P + v] = acc[l];
}

// Column sums of p [rows][cols], into its first row: 64 columns per workgroup,
// the rows dealt to sixteen waves, whose sums are added in order.  For the
// partial sums of many chains over few draws, hundreds of groups of which
// would otherwise be one long chain of loads per lag and coordinate: T = 32,
// 4096 chains, D = 10, six lags 940 -> 22 us.
__global__ void __launch_bounds__(1024)
sum_rows_kernel(double* p, int64_t rows, int64_t cols) {
  __shared__ double sm[16][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t c = (int64_t)blockIdx.x * 64 + lane;
  double s = 0.0;
  if (c < cols) {
#pragma unroll 8
    for (int64_t r = wave; r < rows; r += 16) s += p[r * cols + c];
  }
  sm[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && c < cols) {
#pragma unroll
    for (int w = 1; w < 16; ++w) s += sm[w][lane];
    p[c] = s;
  }
}

// acov[l][d] = sum over the groups and the m side-by-side chains, / T (in place
// where both are 1 and acov is part).
__global__ void __launch_bounds__(256)
autocov_sum_kernel(const double* part, int groups, int n_lags, int m, int D, int64_t T,
                   double* acov) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)n_lags * D) return;
  const int64_t l = i / D;
  const int d = (int)(i - l * D);
  const int64_t P = (int64_t)D * m;
  double s = 0.0;
  const int n = groups * m;   // in order, sixteen loads in flight, then four
  int q = 0;
  auto add = [&](auto count) {
    constexpr int K = decltype(count)::value;
    double v[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int g = (q + k) / m, j = q + k - g * m;
      v[k] = part[((int64_t)g * n_lags + l) * P + (int64_t)j * D + d];
    }
#pragma unroll
    for (int k = 0; k < K; ++k) s += v[k];
    q += K;
  };
  while (q + 16 <= n) add(std::integral_constant<int, 16>{});
  while (q + 4 <= n) add(std::integral_constant<int, 4>{});
  while (q < n) add(std::integral_constant<int, 1>{});
  acov[i] = s / (double)T;
}

int sum_rows(edhmc_ctx* ctx, double* p, int64_t rows, int64_t cols, hipStream_t st) {
  const int64_t wgs = (cols + 63) / 64;
  if (wgs > 2147483647LL) return set_err(ctx, EDHMC_EUNSUPPORTED, "too many columns");
  hipLaunchKernelGGL(sum_rows_kernel, dim3((unsigned)wgs), dim3(1024), 0, st, p, rows, cols);
  return check_launch(ctx, "sum_rows");
}

// scratch: whether the context's may be used (and grow); without it, and where
// the device has no memory for it, the call does without.
// own: the means are made on the way, and written to `mean` unless that is null.
int autocov_lags(edhmc_ctx* ctx, const float* s, int64_t T, int C, int D, int lag0, int n_lags,
                 double* mean, bool own, double* acov, bool scratch, hipStream_t st) {
  AcovArgs a;
  a.s = s;
  a.T = T;
  a.C = C;
  a.D = D;
  a.lag0 = lag0;
  a.n_lags = n_lags;
  a.mean = mean;
  // lags per wave: 8 where there are no more, a quarter of the products and
  // registers of 32 (T = 16, 4096 chains, D = 600, six lags, with the means on
  // the way and no idle waves: 362 -> 92 us)
  const int lags = n_lags <= 8 ? 8 : 32;
  const int lag_blocks = (n_lags + lags - 1) / lags, waves = std::min(kAcWaves, lag_blocks);
  a.lag_wgs = (lag_blocks + waves - 1) / waves;
  auto split = [&](int m, int64_t most) {   // m chains side by side, at most that many groups
    a.m = m;
    a.P = D * m;
    a.blocks = (C + m - 1) / m;
    a.strips = (a.P + 63) / 64;
    const int64_t groups = std::min<int64_t>(most, a.blocks);
    const int64_t per = (a.blocks + groups - 1) / groups;
    a.groups = (int)((a.blocks + per - 1) / per);
  };
  const int m = std::max(1, std::min(C, 64 / D));
  const int64_t most = kAcPartBytes / ((int64_t)D * m * 8);   // lags of one group's partial sums
  if (m > 1 && n_lags > most) {
    for (int64_t l = 0; l < n_lags; l += most)
      EDHMC_TRY(autocov_lags(ctx, s, T, C, D, (int)(lag0 + l), (int)std::min(most, n_lags - l), mean,
                             own, acov + l * D, scratch, st));
    return EDHMC_OK;
  }
  // eight rounds of the 2048 waves that run together, so that the shorter
  // sums of the long lags even out
  const int64_t strips = ((int64_t)D * m + 63) / 64;
  int64_t groups = std::max<int64_t>(1, 16384 / (strips * a.lag_wgs * waves));
  groups = std::min<int64_t>(groups, std::max<int64_t>(1, most / n_lags));
  split(m, groups);
  if (a.m * a.groups == 1) {
    a.part = acov;
  } else if (scratch && dev_reserve(ctx, ctx->acov_part, (size_t)a.groups * n_lags * a.P * 8) == EDHMC_OK) {
    a.part = (double*)ctx->acov_part.p;
  } else {
    split(1, 1);
    a.part = acov;
  }
  const int64_t units = (int64_t)a.strips * a.groups;
  const int64_t grid = (units + 7) / 8 * 8 * a.lag_wgs;
  if (grid > 2147483647LL) return set_err(ctx, EDHMC_EUNSUPPORTED, "autocov: store too wide");
  const dim3 wgs((unsigned)grid), block(64 * waves);
  if (lags == 8 && own) hipLaunchKernelGGL((autocov_kernel<8, true>), wgs, block, 0, st, a);
  else if (lags == 8) hipLaunchKernelGGL((autocov_kernel<8, false>), wgs, block, 0, st, a);
  else if (own) hipLaunchKernelGGL((autocov_kernel<32, true>), wgs, block, 0, st, a);
  else hipLaunchKernelGGL((autocov_kernel<32, false>), wgs, block, 0, st, a);
  EDHMC_TRY(check_launch(ctx, "autocov"));
  // (up to 128 terms autocov_sum_kernel adds them as fast as two launches)
  if (a.groups > 1 && a.groups * a.m > 128) {
    EDHMC_TRY(sum_rows(ctx, a.part, a.groups, (int64_t)n_lags * a.P, st));
    a.groups = 1;
  }
  const int64_t n = (int64_t)n_lags * D;
  hipLaunchKernelGGL(autocov_sum_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                     (const double*)a.part, a.groups, n_lags, a.m, D, T, acov);
  return check_launch(ctx, "autocov_sum");
}

// Draws up to which the direct kernel makes the chain means itself, one pass
// and one launch less (T = 16, 64 chains, D = 100, six lags: 21.4 -> 17.4 us);
// of more draws the moments pass has more loads in flight.
constexpr int64_t kOwnMeanT = 64;

// Lags 0 .. n_lags - 1 and, if asked for, the chain means they take.
int autocov_from_zero(edhmc_ctx* ctx, const float* s, int64_t T, int C, int D, int n_lags,
                      double* mean, double* acov, bool scratch, hipStream_t st) {
  if (T <= kOwnMeanT && !(scratch && autocov_fft_ok(T, n_lags)))
    return autocov_lags(ctx, s, T, C, D, 0, n_lags, mean, true, acov, scratch, st);
  if (!mean && scratch && dev_reserve(ctx, ctx->acov_mean, (size_t)C * D * 8) == EDHMC_OK)
    mean = (double*)ctx->acov_mean.p;
  if (mean && scratch && autocov_fft_ok(T, n_lags)) {
    const int block = autocov_fft_block(T, D);
    int rc = EDHMC_OK;
    for (int d = 0; d < D && rc == EDHMC_OK; d += block)
      rc = autocov_fft(ctx, s, T, C, D, d, std::min(block, D - d), n_lags, mean + d, D, acov + d, D,
                       st);
    if (rc != EDHMC_ENOMEM) return rc;
  }
  if (mean) EDHMC_TRY(launch_moments<float>(ctx, s, T, (int64_t)C * D, 0, mean, nullptr, st));
  return autocov_lags(ctx, s, T, C, D, 0, n_lags, mean, !mean, acov, scratch, st);
}

// A call's turn with the context's readout scratch: it begins when the call
// before has ended, on whatever stream that runs.  Under capture there is none:
// the graph would keep the address of memory that later calls write and grow.
struct ScratchTurn {
  edhmc_ctx* ctx;
  hipStream_t st;
  bool on = false;

  int begin() {
    if (stream_capturing(st)) return EDHMC_OK;
    if (!ctx->acov_used &&
        hipEventCreateWithFlags(&ctx->acov_used, hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();
      ctx->acov_used = nullptr;
      return set_err(ctx, EDHMC_EHIP, "readout: event");
    }
    if (hipStreamWaitEvent(st, ctx->acov_used, 0) != hipSuccess)
      return set_err(ctx, EDHMC_EHIP, "readout: wait");
    on = true;
    return EDHMC_OK;
  }
  int end(int rc) {   // also after an error: something may be running
    if (on && hipEventRecord(ctx->acov_used, st) != hipSuccess && rc == EDHMC_OK)
      return set_err(ctx, EDHMC_EHIP, "readout: event");
    return rc;
  }
};

}  // namespace

namespace edhmc {
int moments_f64(edhmc_ctx* ctx, const double* x, int64_t T, int64_t K, double* mean, double* var,
                hipStream_t st) {
  return launch_moments<double>(ctx, x, T, K, 0, mean, var, st);
}
int sum_rows_f64(edhmc_ctx* ctx, double* p, int64_t rows, int64_t cols, hipStream_t st) {
  return sum_rows(ctx, p, rows, cols, st);
}
}  // namespace edhmc

extern "C" {

int edhmc_sample_moments(edhmc_ctx* ctx, const void* params, int32_t params_dtype, int64_t T,
                         int64_t K, int64_t t0, double* mean_out, double* var_out, void* stream) {
  if (!ctx) return EDHMC_EINVAL;
  DeviceGuard dg(ctx->device);
  if (!params || !mean_out || !var_out || T <= 0 || K <= 0 || t0 < 0 || t0 >= T)
    return set_err(ctx, EDHMC_EINVAL, "bad arguments (T=%lld K=%lld t0=%lld)", (long long)T,
                   (long long)K, (long long)t0);
  if (params_dtype != EDHMC_F32 && params_dtype != 2)
    return set_err(ctx, EDHMC_EINVAL, "params dtype must be fp32 or fp64");
  hipStream_t st = (hipStream_t)stream;
  if (params_dtype == EDHMC_F32)
    return launch_moments<float>(ctx, (const float*)params, T, K, t0, mean_out, var_out, st);
  return launch_moments<double>(ctx, (const double*)params, T, K, t0, mean_out, var_out, st);
}

int edhmc_autocov(edhmc_ctx* ctx, const float* s, int64_t T, int32_t C, int32_t D, int32_t max_lag,
                  double* acov_out, double* chain_mean_out, void* stream) {
  if (!ctx) return EDHMC_EINVAL;
  DeviceGuard dg(ctx->device);
  hipStream_t st = (hipStream_t)stream;
  if (!s || !acov_out || T < 2 || C <= 0 || D <= 0 || max_lag < 0)
    return set_err(ctx, EDHMC_EINVAL, "bad arguments");
  if (max_lag >= T) max_lag = (int)(T - 1);
  ScratchTurn turn{ctx, st};
  EDHMC_TRY(turn.begin());
  return turn.end(autocov_from_zero(ctx, s, T, C, D, max_lag + 1, chain_mean_out, acov_out, turn.on,
                                    st));
}

int edhmc_ess(edhmc_ctx* ctx, const float* s, int64_t T, int32_t C, int32_t D, int32_t between,
              double* ess_out, void* stream) {
  if (!ctx) return EDHMC_EINVAL;
  DeviceGuard dg(ctx->device);
  hipStream_t st = (hipStream_t)stream;
  if (!s || !ess_out || T < 4 || T > 2147483647LL || C <= 0 || D <= 0)
    return set_err(ctx, EDHMC_EINVAL, "bad arguments");
  ScratchTurn turn{ctx, st};
  EDHMC_TRY(turn.begin());
  if (!turn.on) return set_err(ctx, EDHMC_EUNSUPPORTED, "edhmc_ess cannot be captured in a graph");
  auto go = [&]() -> int {
    if (autocov_fft_ok(T, (int)T)) {   // the lags of a block of coordinates at a time
      const int block = autocov_fft_block(T, D);
      EDHMC_TRY(dev_reserve(ctx, ctx->acov_mean, (size_t)C * block * 8));
      EDHMC_TRY(dev_reserve(ctx, ctx->acov, (size_t)T * block * 8));
      double* mean = (double*)ctx->acov_mean.p;
      double* acov = (double*)ctx->acov.p;
      for (int d = 0; d < D; d += block) {
        const int db = std::min(block, D - d);
        EDHMC_TRY(autocov_fft(ctx, s, T, C, D, d, db, (int)T, mean, db, acov, db, st));
        EDHMC_TRY(ess_launch(ctx, acov, mean, T, C, db, between != 0, ess_out + d, st));
      }
      return EDHMC_OK;
    }
    EDHMC_TRY(dev_reserve(ctx, ctx->acov_mean, (size_t)C * D * 8));
    EDHMC_TRY(dev_reserve(ctx, ctx->acov, (size_t)T * D * 8));
    double* mean = (double*)ctx->acov_mean.p;
    double* acov = (double*)ctx->acov.p;
    EDHMC_TRY(autocov_from_zero(ctx, s, T, C, D, (int)T, mean, acov, true, st));
    return ess_launch(ctx, acov, mean, T, C, D, between != 0, ess_out, st);
  };
  return turn.end(go());
}

int edhmc_autocov_lags(edhmc_ctx* ctx, const float* s, int64_t T, int32_t C, int32_t D,
                       int32_t lag0, int32_t n_lags, const double* chain_mean, double* acov_out,
                       void* stream) {
  if (!ctx) return EDHMC_EINVAL;
  DeviceGuard dg(ctx->device);
  if (!s || !acov_out || !chain_mean || T < 2 || C <= 0 || D <= 0 || lag0 < 0 || n_lags <= 0 ||
      (int64_t)lag0 + n_lags > T)
    return set_err(ctx, EDHMC_EINVAL, "bad arguments");
  ScratchTurn turn{ctx, (hipStream_t)stream};
  EDHMC_TRY(turn.begin());
  return turn.end(autocov_lags(ctx, s, T, C, D, lag0, n_lags, (double*)chain_mean, false, acov_out,
                               turn.on, (hipStream_t)stream));
}

}  // extern "C"
