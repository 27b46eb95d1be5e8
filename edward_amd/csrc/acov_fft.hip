// Autocovariances of a sample store s [T, C, D] at all lags, summed over the
// chains (Wiener-Khinchin), and the effective sample sizes from them; FP64.
//
// The sum over the chains goes through: the power spectra of all chains of a
// coordinate are added up, and one inverse transform per coordinate gives its
// lags.  Two chains x, y of a coordinate are transformed as x + i y, zero-padded
// to N >= 2 T - 1 points: |X_k|^2 + |Y_k|^2 = (|Z_k|^2 + |Z_{N-k}|^2) / 2, so
// |Z_k|^2 is summed and made symmetric once.  Rounding is some 1e-15 of the
// lag-0 sum, as for the products summed directly.
//
// T = 1000, C = 1024, D = 256, an effective sample size that needs all lags:
// transpose 440 us (4.8 TB/s), spectra 912, lags back 19, sum 11; direct sums
// in windows of 65, 66, 132, ... lags with the truncation on the host took
// 21 ms (14.9 of them FP64 products).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"
#include "ctx.h"

namespace edhmc {

int moments_f64(edhmc_ctx* ctx, const double* x, int64_t T, int64_t K, double* mean, double* var,
                hipStream_t st);
int sum_rows_f64(edhmc_ctx* ctx, double* p, int64_t rows, int64_t cols, hipStream_t st);

namespace {

struct cplx { double re, im; };
__device__ inline cplx operator+(cplx a, cplx b) { return {a.re + b.re, a.im + b.im}; }
__device__ inline cplx operator-(cplx a, cplx b) { return {a.re - b.re, a.im - b.im}; }
__device__ inline cplx operator*(cplx a, cplx b) {
  return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
__device__ inline cplx mul_mi(cplx a) { return {a.im, -a.re}; }   // times -i

__device__ inline void dft2(cplx& a, cplx& b) {
  const cplx t = a - b;
  a = a + b;
  b = t;
}
// results 0 1 2 3 in a, c, b, d's places: reordered to a b c d
__device__ inline void dft4(cplx& a, cplx& b, cplx& c, cplx& d) {
  dft2(a, c);
  dft2(b, d);
  d = mul_mi(d);
  dft2(a, b);
  dft2(c, d);
  const cplx t = b;
  b = c;
  c = t;
}
__device__ inline void dft8(cplx (&v)[8]) {
  constexpr double h = 0.70710678118654752440;
#pragma unroll
  for (int i = 0; i < 4; ++i) dft2(v[i], v[i + 4]);
  v[5] = cplx{h * (v[5].re + v[5].im), h * (v[5].im - v[5].re)};
  v[6] = mul_mi(v[6]);
  v[7] = cplx{h * (v[7].im - v[7].re), -h * (v[7].re + v[7].im)};
  dft4(v[0], v[1], v[2], v[3]);
  dft4(v[4], v[5], v[6], v[7]);
  const cplx a1 = v[4], a2 = v[1], a3 = v[5], a4 = v[2], a5 = v[6], a6 = v[3];
  v[1] = a1; v[2] = a2; v[3] = a3; v[4] = a4; v[5] = a5; v[6] = a6;
}

// Transform of N = 8^k R points (R = 1: all passes of radix 8) by N / 8
// threads, 8 points each, passes through LDS in natural order (Stockham).
template <int LOG>
struct Fft {
  static constexpr int N = 1 << LOG, TH = N / 8;
  static constexpr int P8 = LOG / 3, R = 1 << (LOG % 3);   // radix-8 passes, radix of the last
  static constexpr int kThreads = TH > 256 ? TH : 256;
  static constexpr int F = kThreads / TH;                  // transforms side by side

  cplx tw[P8 > 1 ? P8 - 1 : 1][7];   // of the passes after the first
  cplx tl[R > 1 ? 8 - 8 / R : 1];    // of the last pass

  // 16-byte element i of a transform: lanes that store 8 Ns apart hit
  // disjoint banks
  static __device__ inline int at(int i) { return i ^ ((i >> 3) & 15); }

  __device__ inline void init(int j) {
    auto w = [](int k, int n) {   // exp(-2 pi i k / n)
      cplx c;
      sincospi(-2.0 * k / n, &c.im, &c.re);
      return c;
    };
    int ns = 8;
#pragma unroll
    for (int p = 1; p < P8; ++p, ns *= 8)
#pragma unroll
      for (int r = 1; r < 8; ++r) tw[p - 1][r - 1] = w((j % ns) * r, 8 * ns);
    if constexpr (R > 1) {
#pragma unroll
      for (int m = 0; m < 8 / R; ++m)
#pragma unroll
        for (int r = 1; r < R; ++r) tl[m * (R - 1) + r - 1] = w((j + m * TH) * r, N);
    }
  }
  // v[r] = element j + r TH of the input; on return v[i] is element
  // out(j, i) of the transform
  static __device__ inline int out(int j, int i) {
    return R > 1 ? j + (i / R) * TH + (i % R) * (N / R) : j + i * TH;
  }
  __device__ inline void run(cplx (&v)[8], cplx* lds, int j) const {
    int ns = 1;
#pragma unroll
    for (int p = 0; p < P8; ++p, ns *= 8) {
      if (p > 0)
#pragma unroll
        for (int r = 1; r < 8; ++r) v[r] = v[r] * tw[p - 1][r - 1];
      dft8(v);
      if (p == P8 - 1 && R == 1) break;
      __syncthreads();   // everybody has read the pass before
      const int d = (j / ns) * ns * 8 + j % ns;
#pragma unroll
      for (int r = 0; r < 8; ++r) lds[at(d + r * ns)] = v[r];
      __syncthreads();
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = lds[at(p == P8 - 1 ? out(j, i) : j + i * TH)];
    }
    if constexpr (R > 1) {
#pragma unroll
      for (int m = 0; m < 8 / R; ++m)
#pragma unroll
        for (int r = 1; r < R; ++r) v[m * R + r] = v[m * R + r] * tl[m * (R - 1) + r - 1];
#pragma unroll
      for (int m = 0; m < 8 / R; ++m) {
        if constexpr (R == 2) dft2(v[2 * m], v[2 * m + 1]);
        else dft4(v[4 * m], v[4 * m + 1], v[4 * m + 2], v[4 * m + 3]);
      }
    }
  }
};

// The series of kc / db chains and db coordinates, chains D columns of s
// [T][K] apart, as rows of st [kc][Tp], and their means [chain][ldm].
__global__ void __launch_bounds__(256)
acov_rows_kernel(const float* __restrict__ s, int64_t T, int64_t K, int D, int64_t kc, int db,
                 int64_t Tp, float* __restrict__ st, double* __restrict__ mean, int64_t ldm) {
  __shared__ float tile[64][65];
  __shared__ double sum[4][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t c0 = (int64_t)blockIdx.x * 64;
  const int col = (int)min(c0 + lane, kc - 1), chain = col / db, d = col - chain * db;
  const float* p = s + (int64_t)chain * D + d;
  float v[16];
  auto load = [&](int64_t t0) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int64_t t = t0 + 16 * wave + i;
      v[i] = t < T ? p[t * K] : 0.0f;
    }
  };
  double a = 0.0;
  load(0);
  for (int64_t t0 = 0; t0 < T; t0 += 64) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      a += (double)v[i];
      tile[lane][16 * wave + i] = v[i];
    }
    __syncthreads();
    if (t0 + 64 < T) load(t0 + 64);
    if (t0 + lane < T) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int64_t c = c0 + 16 * wave + i;
        if (c < kc) st[c * Tp + t0 + lane] = tile[16 * wave + i][lane];
      }
    }
    __syncthreads();
  }
  sum[wave][lane] = a;
  __syncthreads();
  if (wave == 0 && c0 + lane < kc)
    mean[chain * ldm + d] = (((sum[0][lane] + sum[1][lane]) + sum[2][lane]) + sum[3][lane]) / (double)T;
}

// Power spectra of the chain pairs of coordinate d, one workgroup per d and
// group of pairs, F pairs at a time; added to part [groups F][D][N] (the first
// chunk of chains: stored there).  131,072 pairs of 2048 points: 912 us, 13
// TF, two waves per SIMD waiting for each other's LDS passes; the twiddles
// stay in registers (three waves per SIMD spill: 1532 us).
template <int LOG>
__global__ void __launch_bounds__(Fft<LOG>::kThreads)
acov_power_kernel(const float* __restrict__ st, int64_t T, int64_t Tp, int D, int chains,
                  const double* __restrict__ mean, int64_t ldm, int groups, bool first,
                  double* __restrict__ part) {
  using X = Fft<LOG>;
  __shared__ __align__(16) cplx lds[X::F * X::N];
  const int d = blockIdx.x % D, g = blockIdx.x / D;
  const int slot = threadIdx.x / X::TH, j = threadIdx.x % X::TH;
  X fft;
  fft.init(j);
  double acc[8];
  double* out = part + (((int64_t)g * X::F + slot) * D + d) * X::N;
#pragma unroll
  for (int i = 0; i < 8; ++i) acc[i] = first ? 0.0 : out[X::out(j, i)];
  const int pairs = (chains + 1) / 2, step = groups * X::F;
  float xr[4], yr[4];
  auto fetch = [&](int q) {   // the series' draws fill the lower half of the points
    const int c = 2 * (q + slot);
    const float* x = st + ((int64_t)c * D + d) * Tp;
    const float* y = x + (int64_t)D * Tp;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = j + i * X::TH;
      xr[i] = c < chains && t < T ? x[t] : 0.0f;
      yr[i] = c + 1 < chains && t < T ? y[t] : 0.0f;
    }
  };
  fetch(g * X::F);
  for (int q = g * X::F; q < pairs; q += step) {
    const int c = 2 * (q + slot);
    const double mx = c < chains ? mean[c * ldm + d] : 0.0;
    const double my = c + 1 < chains ? mean[(c + 1) * ldm + d] : 0.0;
    cplx v[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool in = j + i * X::TH < T;
      v[i].re = in ? (double)xr[i] - mx : 0.0;
      v[i].im = in ? (double)yr[i] - my : 0.0;
      v[i + 4] = cplx{0.0, 0.0};
    }
    if (q + step < pairs) fetch(q + step);
    fft.run(v, lds + slot * X::N, j);
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] += v[i].re * v[i].re + v[i].im * v[i].im;
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) out[X::out(j, i)] = acc[i];
}

// acov[l * ld + d] = sum over the parts, made symmetric, transformed back, / (N T).
template <int LOG>
__global__ void __launch_bounds__(Fft<LOG>::kThreads)
acov_lags_kernel(const double* __restrict__ part, int parts, int D, int64_t T, int n_lags,
                 double* __restrict__ acov, int64_t ld) {
  using X = Fft<LOG>;
  __shared__ __align__(16) cplx lds[X::F * X::N];
  const int slot = threadIdx.x / X::TH, j = threadIdx.x % X::TH;
  const int d = blockIdx.x * X::F + slot;
  const bool ok = d < D;
  X fft;
  fft.init(j);
  double p[8], m[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) p[i] = m[i] = 0.0;
  for (int q = 0; q < parts; ++q) {
    const double* in = part + ((int64_t)q * D + (ok ? d : 0)) * X::N;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int k = j + i * X::TH;
      p[i] += in[k];
      m[i] += in[(X::N - k) & (X::N - 1)];
    }
  }
  cplx v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = cplx{0.5 * (p[i] + m[i]), 0.0};
  fft.run(v, lds + slot * X::N, j);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int l = X::out(j, i);
    if (ok && l < n_lags) acov[l * ld + d] = v[i].re / X::N / (double)T;
  }
}

// Effective sample size of each coordinate from the sums over C chains of the
// autocovariances at all T lags: within- and (spread, or null: none)
// between-chain variance, Geyer's initial positive and monotone sequence.  A
// wave per coordinate, 64 pairs of lags at a time (a thread per coordinate
// that walks them: 137 us at T = 1000, D = 256, here 11).
__global__ void __launch_bounds__(64)
ess_kernel(const double* __restrict__ acov, const double* __restrict__ spread, int64_t T, int C,
           int D, double floor_tau, double* __restrict__ ess) {
  const int d = blockIdx.x, lane = threadIdx.x;
  const double n = (double)T, M = (double)C;
  const double W = acov[d] / M * n / (n - 1.0);
  const double var = W * (n - 1.0) / n + (spread ? spread[d] * (M / (M - 1.0)) : 0.0);
  if (!(var > 0.0)) {   // no movement: nothing was sampled
    if (lane == 0) ess[d] = 0.0;
    return;
  }
  double total = 0.0, low = 0.0;
  const int64_t pairs = T / 2;
  for (int64_t i0 = 0; i0 < pairs; i0 += 64) {
    const int64_t i = i0 + lane;
    double p = 0.0;   // past the end: stops
    if (i < pairs) {
      const double r0 = i == 0 ? 1.0 : 1.0 - (W - acov[2 * i * D + d] / M) / var;
      p = r0 + (1.0 - (W - acov[(2 * i + 1) * D + d] / M) / var);
    }
    const uint64_t stop = __ballot(p <= 0.0);
    const int first = stop ? __builtin_ctzll(stop) : 64;
    // running minimum over the lanes, then with the pairs before
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const double q = __shfl_up(p, off, 64);
      if (lane >= off) p = fmin(p, q);
    }
    if (i0 > 0) p = fmin(p, low);
    low = __shfl(p, 63, 64);
    double s = lane < first ? p : 0.0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    total += s;
    if (first < 64) break;
  }
  if (lane == 0) ess[d] = M * n / fmax(-1.0 + 2.0 * total, floor_tau);
}

constexpr int64_t kStoreBytes = 256 << 20;   // transposed chains held at a time
constexpr int64_t kPartBytes = 64 << 20;     // partial spectra

// Spectra of a coordinate, F side by side: 16 KB, 32 from 1025 draws on.
template <int LOG>
constexpr int64_t spectra_bytes = (int64_t)Fft<LOG>::F * Fft<LOG>::N * 8;

// Coordinates s points at the first of; D: coordinates of the store.
template <int LOG>
int launch(edhmc_ctx* ctx, const float* s, int64_t T, int C, int D, int db, int n_lags,
           double* mean, int64_t ldm, double* acov, int64_t ld, hipStream_t st) {
  using X = Fft<LOG>;
  const int64_t Tp = (T + 15) / 16 * 16;
  // an even number of chains at a time
  int64_t chunk = std::max<int64_t>(2, kStoreBytes / (Tp * 4 * db)) & ~1LL;
  chunk = std::min<int64_t>(chunk, C);
  const int64_t sets = ((chunk + 1) / 2 + X::F - 1) / X::F;   // of F pairs
  int64_t groups = std::max<int64_t>(1, 4096 / db);           // two rounds of eight per unit
  groups = std::min(groups, std::max<int64_t>(1, kPartBytes / (db * spectra_bytes<LOG>)));
  groups = std::min(groups, sets);
  EDHMC_TRY(dev_reserve(ctx, ctx->acov_rows, (size_t)(chunk * db * Tp) * 4));
  EDHMC_TRY(dev_reserve(ctx, ctx->acov_part, (size_t)(groups * db * spectra_bytes<LOG>)));
  float* rows = (float*)ctx->acov_rows.p;
  double* part = (double*)ctx->acov_part.p;
  for (int64_t c0 = 0; c0 < C; c0 += chunk) {
    const int64_t cc = std::min<int64_t>(chunk, C - c0), kc = cc * db;
    hipLaunchKernelGGL(acov_rows_kernel, dim3((unsigned)((kc + 63) / 64)), dim3(256), 0, st,
                       s + c0 * D, T, (int64_t)C * D, D, kc, db, Tp, rows, mean + c0 * ldm, ldm);
    EDHMC_TRY(check_launch(ctx, "acov_rows"));
    hipLaunchKernelGGL((acov_power_kernel<LOG>), dim3((unsigned)(groups * db)), dim3(X::kThreads),
                       0, st, (const float*)rows, T, Tp, db, (int)cc,
                       (const double*)mean + c0 * ldm, ldm, (int)groups, c0 == 0, part);
    EDHMC_TRY(check_launch(ctx, "acov_power"));
  }
  int parts = (int)(groups * X::F);
  // many chains of few coordinates: too long a chain of loads for the few
  // workgroups of the next kernel (T = 100, 4096 chains, D = 10, effective
  // sample sizes: 1470 -> 97 us; with 16 parts both are alike)
  if (parts > 16) {
    EDHMC_TRY(sum_rows_f64(ctx, part, parts, (int64_t)db * X::N, st));
    parts = 1;
  }
  hipLaunchKernelGGL((acov_lags_kernel<LOG>), dim3((db + X::F - 1) / X::F), dim3(X::kThreads), 0,
                     st, (const double*)part, parts, db, T, n_lags, acov, ld);
  return check_launch(ctx, "acov_lags");
}

template <typename F>
auto with_log(int64_t T, F f) {
  using std::integral_constant;
  if (T <= 64) return f(integral_constant<int, 7>{});
  if (T <= 128) return f(integral_constant<int, 8>{});
  if (T <= 256) return f(integral_constant<int, 9>{});
  if (T <= 512) return f(integral_constant<int, 10>{});
  if (T <= 1024) return f(integral_constant<int, 11>{});
  return f(integral_constant<int, 12>{});
}

}  // namespace

constexpr int64_t kFftMaxT = 2048;   // 4096 points of 16 bytes in LDS

// From 33 lags on, where the direct kernel takes a second block of 32.  us of a
// call, 32 lags directly / 64 directly / all here: T = 1000, C = 1024, D = 256
// 723 / 1165 / 1281; T = 2000, 1024, 128 718 / 1165 / 1678; T = 200, 1024, 256
// 180 / 300 / 271; T = 100, 4096, 10 62 / 68 / 60; T = 1000, one chain, D = 10
// 178 / 219 / 36.  (Up to 64 lags of long chains in a wide store the direct
// kernel would still be ahead.)
bool autocov_fft_ok(int64_t T, int n_lags) { return T <= kFftMaxT && n_lags > 32; }

// Coordinates a call takes: as many as leave the transposed chains (two at
// least) and the spectra (one group) within their bytes, in equal blocks.
int autocov_fft_block(int64_t T, int D) {
  const int64_t spec = with_log(T, [](auto lg) { return spectra_bytes<decltype(lg)::value>; });
  const int64_t most = std::min(kPartBytes / spec, kStoreBytes / (2 * 4 * ((T + 15) / 16 * 16)));
  const int64_t blocks = (D + most - 1) / most;
  return (int)((D + blocks - 1) / blocks);
}

// Coordinates d0 .. d0 + db - 1, at most a block: their lags to acov [n_lags][ld]
// and means to mean [C][ldm].
int autocov_fft(edhmc_ctx* ctx, const float* s, int64_t T, int C, int D, int d0, int db, int n_lags,
                double* mean, int64_t ldm, double* acov, int64_t ld, hipStream_t st) {
  return with_log(T, [&](auto lg) {
    return launch<decltype(lg)::value>(ctx, s + d0, T, C, D, db, n_lags, mean, ldm, acov, ld, st);
  });
}

int ess_launch(edhmc_ctx* ctx, const double* acov, const double* mean, int64_t T, int C, int D,
               bool between, double* ess, hipStream_t st) {
  double* var = nullptr;
  if (between && C > 1) {
    EDHMC_TRY(dev_reserve(ctx, ctx->ess_spread, (size_t)D * 16));
    double* m = (double*)ctx->ess_spread.p;
    var = m + D;
    EDHMC_TRY(moments_f64(ctx, mean, C, D, m, var, st));
  }
  const double floor_tau = 1.0 / log10((double)C * (double)T);
  hipLaunchKernelGGL(ess_kernel, dim3(D), dim3(64), 0, st, acov, (const double*)var, T,
                     C, D, floor_tau, ess);
  return check_launch(ctx, "ess");
}

}  // namespace edhmc
