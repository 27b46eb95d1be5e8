// Newton terms of the GLM log joint at one position: log p, gradient and
// the negative Hessian P = X^T diag(s) X + diag(1 / scale^2), where s_n is
// the likelihood's curvature in eta_n (Bernoulli: sigma (1 - sigma);
// Normal: 1 / lik_scale^2).  These drive a Newton / Laplace warm start of
// the chains (the mode and the Gaussian approximation N(mode, P^-1) of the
// Laplace approximation, edward/inferences/laplace.py:17-137).
//
// Kernels (X as bound: row-major [N_pad, D_pad], fp32 or bf16):
//   newton_rows_kernel  a wave takes eight rows: eta = x.w (fp32 FMA, a lane
//                       holds 8 consecutive columns), r = dll/deta, s, FP64
//                       log-lik partial per workgroup.  Bound by the read of X:
//                       207 us at N = 1M, D = 512, bf16 (one row at a time,
//                       waiting for its reduction and its exp and log1p: 505).
//   newton_gram_kernel  blocks of sum_n s_n x_n x_n^T over a slice of the rows
//                       on the fp32 matrix cores; the diagonal blocks also sum
//                       r_n x_n (the gradient).  fp32 partials per slice.
//   newton_final_kernel FP64 sum of the slice partials, prior terms.
// Work: 2 N D_pad^2 flop for the Gram matrix, one read of X for the rows.
#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>

#include "common.h"
#include "ctx.h"
#include "../../include/edhmc.h"

using namespace edhmc;

namespace {

constexpr int kGramSlices = 64;    // row slices (split of the row sum)

template <typename T>
__device__ inline float load_x(const T* p);
template <>
__device__ inline float load_x<float>(const float* p) { return *p; }
template <>
__device__ inline float load_x<bf16_t>(const bf16_t* p) { return bf16_to_f32(*p); }

template <typename T>
__global__ void __launch_bounds__(256)
newton_rows_kernel(const T* __restrict__ X, const float* __restrict__ y, int64_t N, int D_pad,
                   const float* __restrict__ w, LikParams lp, float* __restrict__ r_out,
                   float* __restrict__ s_out, double* __restrict__ ll_part) {
  extern __shared__ float w_lds[];   // [D_pad]
  __shared__ double red[4];
  for (int d = threadIdx.x; d < D_pad; d += 256) w_lds[d] = w[d];
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double ll = 0.0;
  for (int64_t n0 = ((int64_t)blockIdx.x * 4 + wave) * 8; n0 < N; n0 += (int64_t)gridDim.x * 32) {
    float acc[8] = {};
    for (int d0 = lane * 8; d0 < D_pad; d0 += 512) {
      T x[8][8];
      float wv[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {   // rows past N: the last one's, not used
        const T* row = X + min(n0 + i, N - 1) * D_pad + d0;
        __builtin_memcpy(x[i], __builtin_assume_aligned(row, 16), sizeof(x[i]));
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) wv[e] = w_lds[d0 + e];
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[i] = fmaf(load_x(&x[i][e]), wv[e], acc[i]);
    }
    // sums over the lanes, lane bit 5 first; each step halves the rows a lane
    // is still adding, down to row n0 + (lane >> 3)
#pragma unroll
    for (int k = 4; k > 0; k >>= 1) {
      const bool up = lane & (8 * k);
#pragma unroll
      for (int i = 0; i < k; ++i) {
        const float send = up ? acc[i] : acc[i + k], keep = up ? acc[i + k] : acc[i];
        acc[i] = keep + __shfl_xor(send, 8 * k, 64);
      }
    }
#pragma unroll
    for (int off = 4; off > 0; off >>= 1) acc[0] += __shfl_xor(acc[0], off, 64);
    const int64_t n = n0 + (lane >> 3);
    if ((lane & 7) == 0 && n < N) {
      const float eta = acc[0], yv = y[n];
      float dll, s;
      double l;
      if (lp.lik == LIK_BERNOULLI) {
        const double e = exp(-fabs((double)eta));
        const double sig = eta >= 0.0f ? 1.0 / (1.0 + e) : e / (1.0 + e);
        dll = (float)((double)yv - sig);
        s = (float)(sig * (1.0 - sig));
        l = (double)yv * eta - (fmax((double)eta, 0.0) + log1p(e));
      } else {
        const double dd = (double)yv - eta;
        dll = (float)(dd * lp.inv_s2);
        s = lp.inv_s2;
        l = -0.5 * dd * dd * lp.inv_s2 + lp.ll_const;
      }
      r_out[n] = dll;
      s_out[n] = s;
      ll += l;
    }
  }
  ll = block_sum_f64<256>(ll, red);
  if (threadIdx.x == 0) ll_part[blockIdx.x] = ll;
}

constexpr int gram_threads(int BT, int WT) { return BT / WT * (BT / WT) * 64; }

// One BT x BT block of sum_n s_n x_n x_n^T over a slice of the rows, waves of
// WT x WT; the diagonal blocks also sum r_n x_n.  32x32x2 fp32 matrix
// instructions: chains of fused multiply-adds in k order, so every sum runs
// over the slice's rows in order, with the factor s_n x_ni rounded first (P_ij
// and P_ji differ in that factor: both are computed).
//
// Rows are staged KR at a time as fp32, scaled and plain, the next ones loaded
// while these are multiplied; column c of an odd row sits at c ^ 32, so that
// the two rows of an operand read hit different banks.
//
// Bound: the matrix instructions, 2 N D_pad^2 operations, 0.86 of the cycles.
// N = 1M, D = 512, bf16 X: 10.7 ms with vector FMAs -> 4.2 (124 TF).  One
// workgroup of sixteen waves per compute unit keeps its four waves per SIMD
// in step (four workgroups of four drift apart and the last ones run alone:
// 4.55 ms); staging sits between the halves of a stage's products so that no
// wave comes to the barrier with it still to do (after them: 4.31).
template <typename T, int BT, int WT>
__global__ void __launch_bounds__(gram_threads(BT, WT), 4)
newton_gram_kernel(const T* __restrict__ X, int64_t N, int D_pad, const float* __restrict__ r,
                   const float* __restrict__ s, int64_t rows_per, float* __restrict__ H_part,
                   float* __restrict__ g_part) {
  constexpr int NT = gram_threads(BT, WT);
  constexpr int KR = NT * 8 / BT;          // rows per stage
  constexpr int E = 16 / sizeof(T);        // elements per load
  constexpr int CH = 8 / E;                // loads per thread and operand
  constexpr int WW = BT / WT, MT = WT / 32;   // waves per side; 32 x 32 blocks per wave, each way
  __shared__ __align__(16) float A[2][KR * BT], B[2][KR * BT];
  __shared__ float Rv[2][KR];
  const int nb = D_pad / BT, tiles = nb * nb;
  // a slice's blocks run on one XCD and share its rows in L2
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int slice = xcd + 8 * (local / tiles), tile = local % tiles;
  const int bi = tile / nb, bj = tile % nb;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wi = wave / WW, wj = wave % WW, l32 = lane & 31, hi = lane >> 5;
  const int64_t n_lo = (int64_t)slice * rows_per;
  const int64_t n_hi = n_lo + rows_per < N ? n_lo + rows_per : N;
  const bool diag = bi == bj;
  f32x16_t acc[MT][MT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
  float gacc = 0.0f;   // gradient of column bi BT + tid (diagonal blocks, first BT threads)

  uint4 av[CH], bv[CH];
  float sv[CH], rv = 0.0f;
  auto load = [&](int64_t n0) {
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int q = i * NT + tid, row = q / (BT / E), c = (q % (BT / E)) * E;
      const int64_t n = n0 + row;
      const bool ok = n < n_hi;
      av[i] = bv[i] = make_uint4(0, 0, 0, 0);
      sv[i] = 0.0f;
      if (ok) {
        av[i] = *(const uint4*)(X + n * D_pad + bi * BT + c);
        bv[i] = *(const uint4*)(X + n * D_pad + bj * BT + c);
        sv[i] = s[n];
      }
    }
    if (diag && tid < KR) rv = n0 + tid < n_hi ? r[n0 + tid] : 0.0f;
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int q = i * NT + tid, row = q / (BT / E), c = (q % (BT / E)) * E;
      const int at = row * BT + (c ^ ((row & 1) * 32));
      const T* a = (const T*)&av[i];
      const T* b = (const T*)&bv[i];
#pragma unroll
      for (int e = 0; e < E; e += 4) {
        float4 x, y;
        x.x = load_x(a + e) * sv[i];
        x.y = load_x(a + e + 1) * sv[i];
        x.z = load_x(a + e + 2) * sv[i];
        x.w = load_x(a + e + 3) * sv[i];
        y.x = load_x(b + e);
        y.y = load_x(b + e + 1);
        y.z = load_x(b + e + 2);
        y.w = load_x(b + e + 3);
        *(float4*)&A[buf][at + e] = x;
        *(float4*)&B[buf][at + e] = y;
      }
    }
    if (diag && tid < KR) Rv[buf][tid] = rv;
  };
  auto multiply = [&](int buf, int k0) {   // half a stage
#pragma unroll
    for (int k = k0; k < k0 + KR / 2; k += 2) {
      float a[MT], b[MT];
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        // columns wi WT + 32 i + l32 of an odd row: at ^ 32
        const int ca = wi * WT + 32 * i, cb = wj * WT + 32 * i;
        a[i] = A[buf][(k + hi) * BT + ((ca ^ (hi * 32)) + l32)];
        b[i] = B[buf][(k + hi) * BT + ((cb ^ (hi * 32)) + l32)];
      }
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
    }
  };
  auto gradient = [&](int buf) {
    if (diag && tid < BT) {
#pragma unroll 8
      for (int k = 0; k < KR; ++k) gacc = fmaf(Rv[buf][k], B[buf][k * BT + (tid ^ ((k & 1) * 32))], gacc);
    }
  };
  if (n_lo < n_hi) {
    load(n_lo);
    stage(0);
    load(n_lo + KR);
    __syncthreads();
    int buf = 0;
    for (int64_t n0 = n_lo; n0 < n_hi; n0 += KR) {
      multiply(buf, 0);
      stage(buf ^ 1);
      gradient(buf);
      multiply(buf, KR / 2);
      load(n0 + 2 * KR);
      __syncthreads();
      buf ^= 1;
    }
  }
  float* out = H_part + (int64_t)slice * D_pad * D_pad;
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int a = bi * BT + wi * WT + 32 * i + (v & 3) + 8 * (v >> 2) + 4 * hi;
        const int b = bj * BT + wj * WT + 32 * j + l32;
        out[(int64_t)a * D_pad + b] = acc[i][j][v];
      }
  if (diag && tid < BT) g_part[(int64_t)slice * D_pad + bi * BT + tid] = gacc;
}

// P[i][j] = sum of slices + [i == j] / scale_i^2; grad_i = sum of slices -
// (w_i - loc_i) / scale_i^2; logp = sum of ll partials + prior (FP64).
__global__ void __launch_bounds__(256)
newton_final_kernel(const float* __restrict__ H_part, const float* __restrict__ g_part,
                    const double* __restrict__ ll_part, int n_ll, int D, int D_pad,
                    const float* __restrict__ w, const float* __restrict__ ploc,
                    const float* __restrict__ pscale, double* __restrict__ logp_out,
                    double* __restrict__ grad_out, double* __restrict__ P_out) {
  __shared__ double red[4];
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < (int64_t)D * D) {
    const int a = (int)(i / D), b = (int)(i - (int64_t)a * D);
    double v = 0.0;
    for (int q = 0; q < kGramSlices; ++q) v += H_part[(int64_t)q * D_pad * D_pad + (int64_t)a * D_pad + b];
    if (a == b) v += 1.0 / ((double)pscale[a] * (double)pscale[a]);
    P_out[i] = v;
  }
  if (blockIdx.x == 0) {
    double lp = 0.0;
    for (int d = threadIdx.x; d < D; d += 256) {
      double g = 0.0;
      for (int q = 0; q < kGramSlices; ++q) g += g_part[(int64_t)q * D_pad + d];
      const double sc = pscale[d], t = ((double)w[d] - (double)ploc[d]) / sc;
      grad_out[d] = g - t / sc;
      lp += -0.5 * t * t - log(sc) - 0.5 * kLog2Pi;
    }
    for (int q = threadIdx.x; q < n_ll; q += 256) lp += ll_part[q];
    lp = block_sum_f64<256>(lp, red);
    if (threadIdx.x == 0) *logp_out = lp;
  }
}

}  // namespace

extern "C" int edhmc_newton_terms(edhmc_ctx* ctx, const float* w, double* logp_out,
                                  double* grad_out, double* neg_hess_out, void* stream) {
  if (!ctx) return EDHMC_EINVAL;
  DeviceGuard dg(ctx->device);
  if (!ctx->bound) return set_err(ctx, EDHMC_ESTATE, "no model bound");
  if (ctx->hier) return set_err(ctx, EDHMC_EUNSUPPORTED, "Newton terms are for the GLM");
  if (ctx->has_kinds)
    return set_err(ctx, EDHMC_EUNSUPPORTED, "Newton terms need Normal priors on every coordinate");
  if (!w || !logp_out || !grad_out || !neg_hess_out)
    return set_err(ctx, EDHMC_EINVAL, "NULL argument");
  // the likelihood weight multiplies the data terms (it is 1 for HMC)
  if (ctx->lik_weight != 1.0f)
    return set_err(ctx, EDHMC_EUNSUPPORTED, "Newton terms need likelihood weight 1");
  hipStream_t st = (hipStream_t)stream;
  const int D = ctx->D, D_pad = ctx->D_pad;
  const int64_t N = ctx->N;
  const int rows_grid = 2048;
  const int64_t rows_per = (N + kGramSlices - 1) / kGramSlices;
  // scratch: r and s [N_pad], slice partials of P and the gradient, log-lik
  // partials, the padded position
  const size_t rs_bytes = (size_t)ctx->N_pad * 8;
  const size_t h_bytes = (size_t)kGramSlices * D_pad * D_pad * 4;
  const size_t g_bytes = (size_t)kGramSlices * D_pad * 4;
  const size_t ll_bytes = (size_t)rows_grid * 8;
  const size_t w_bytes = (size_t)D_pad * 4;
  EDHMC_TRY(dev_alloc(ctx, ctx->newton, rs_bytes + h_bytes + g_bytes + ll_bytes + w_bytes, false));
  char* base = (char*)ctx->newton.p;
  float* r = (float*)base;
  float* s = r + ctx->N_pad;
  float* H = (float*)(base + rs_bytes);
  float* g = (float*)(base + rs_bytes + h_bytes);
  double* ll = (double*)(base + rs_bytes + h_bytes + g_bytes);
  float* wp = (float*)(base + rs_bytes + h_bytes + g_bytes + ll_bytes);
  if (hipMemsetAsync(wp, 0, w_bytes, st) != hipSuccess ||
      hipMemcpyAsync(wp, w, (size_t)D * 4, hipMemcpyDeviceToDevice, st) != hipSuccess)
    return set_err(ctx, EDHMC_EHIP, "newton: copy of w failed");
  LikParams lp;
  lp.lik = ctx->lik;
  lp.inv_s2 = 1.0f / (ctx->lik_scale * ctx->lik_scale);
  lp.ll_const = -log((double)ctx->lik_scale) - 0.5 * kLog2Pi;
  const size_t shm = (size_t)D_pad * 4;
  auto terms = [&](auto t) {
    using T = decltype(t);
    const T* X = (const T*)ctx->Xr.p;
    hipLaunchKernelGGL(newton_rows_kernel<T>, dim3(rows_grid), dim3(256), shm, st, X,
                       (const float*)ctx->y.p, N, D_pad, wp, lp, r, s, ll);
    auto gram = [&](auto bt, auto wt) {
      constexpr int BT = decltype(bt)::value, WT = decltype(wt)::value;
      const int nb = D_pad / BT;
      hipLaunchKernelGGL((newton_gram_kernel<T, BT, WT>), dim3(nb * nb * kGramSlices),
                         dim3(gram_threads(BT, WT)), 0, st, X, N, D_pad, r, s, rows_per, H, g);
    };
    // Sixteen waves on 256 x 256 or 128 x 128 where the 64 slices' blocks then
    // still fill the card; four on 64 x 64 otherwise.  N = 200,001, whole call:
    // D = 256 455 us for 551 with 64 x 64 blocks, D = 512 1393 for 1490 with
    // 128 x 128 of four waves, D = 100 309 for 500 with 128 x 128.
    using std::integral_constant;
    if (D_pad % 256 == 0 && D_pad >= 512)
      gram(integral_constant<int, 256>{}, integral_constant<int, 64>{});
    else if (D_pad % 128 == 0 && D_pad >= 256)
      gram(integral_constant<int, 128>{}, integral_constant<int, 32>{});
    else
      gram(integral_constant<int, 64>{}, integral_constant<int, 32>{});
  };
  if (ctx->cdt == EDHMC_BF16) terms(bf16_t{});
  else terms(float{});
  EDHMC_TRY(check_launch(ctx, "newton_gram"));
  hipLaunchKernelGGL(newton_final_kernel, dim3((unsigned)(((int64_t)D * D + 255) / 256)),
                     dim3(256), 0, st, H, g, ll, rows_grid, D, D_pad, wp,
                     (const float*)ctx->ploc.p, (const float*)ctx->pscale.p, logp_out, grad_out,
                     neg_hess_out);
  return check_launch(ctx, "newton_final");
}
