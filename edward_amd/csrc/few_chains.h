// One-pass gradient of the GLM for up to kFewMax chains in fp32, D <= 256:
// both products of a gradient evaluation,
//   eta[n, c] = x_n . w_c,   G[c, d] = sum_n r(eta[n, c], y_n) x_n[d],
// from one read of X, the residuals never leaving the registers.
//
// A workgroup of four waves owns a contiguous range of data rows, streamed
// through LDS in tiles of 64 RB rows, 16 RB per wave.  Every wave keeps the
// positions (the matrix cores' 16 columns, zero past the last chain) and its
// gradient sums in registers for the whole range.  Per 16-row block
//   GEMM1  v_mfma_f32_16x16x4_f32 with A = X (16 rows), B = W^T: lane l holds
//          chain l & 15, and its four results are rows 4 (l >> 4) + v;
//   epilogue  the residual (and, with LL, the log-likelihood term) of those
//          four elements, in place;
//   GEMM2  the residuals are already the A operand of the second product
//          (chain l & 15, k = l >> 4): MFMA v covers the rows
//          {4 h + v : h < 4}, with B = X of those rows from the same tile.
// G is summed per wave over its rows in fp32, the waves of a workgroup in a
// fixed order through LDS, and the row ranges by the chain kernels (fixed
// order: the same bits on every run).
//
// What bounds it: the read of X (N = 581,012 rows of 64 columns, 149 MB: 31
// us, 4.7 TB/s, what a large copy reaches here; the matrix cores are busy for
// half of that time).  So X is kept with its columns rounded to 16 below 64
// (N = 1e6, D = 10: 64 MB instead of 256).
#pragma once

#include "common.h"
#include "ctx.h"

namespace edhmc {

constexpr int kFewTile = 16;       // chain columns of the matrix instruction
constexpr int kFewWaves = 4;
constexpr int kFewThreads = 64 * kFewWaves;

struct FewArgs {
  const float* X;          // [N_pad][DP] row-major, zero past D columns and N rows
  const float* y;          // [N_pad], zero past N
  const float* W;          // positions, rows ldw floats apart, zero past D columns
  int64_t ldw;
  int64_t N;
  int64_t rows_per_split;  // multiple of 64 RB
  int C, splits;           // chains (<= kFewTile), row ranges
  LikParams lp;
  float* Gpart;            // [splits][C][ldg]
  int64_t ldg;
  double* llpart;          // [splits][ll_ld]
  int64_t ll_ld;
};

// 16-row blocks per wave and tile: tiles of about 16 KB.
constexpr int few_rb(int DP) { return DP <= 16 ? 4 : DP <= 32 ? 2 : 1; }
// Whole tiles of X and y are read: N_pad is a multiple of the longest one.
constexpr int kFewRows = 16 * few_rb(16) * kFewWaves;

template <int DP, bool GRAD, bool LL>
__global__ void __launch_bounds__(kFewThreads) __attribute__((amdgpu_waves_per_eu(1)))
few_chains_kernel(FewArgs a) {
  constexpr int NT = kFewThreads, RB = few_rb(DP), TR = 16 * RB * kFewWaves;
  constexpr int S = DP + 4;                 // LDS row stride (floats), 4 or 20 mod 32: the 16
                                            // rows of a b128 read hit disjoint banks
  constexpr int Q = DP / 16;                // 16-column chunks of GEMM1
  // column groups of GEMM2, by the width of the B operand's LDS read
  constexpr int G4 = DP / 64, G2 = DP % 64 / 32, G1 = DP % 32 / 16;
  constexpr int NG = DP / 16;               // accumulators (16 columns each)
  constexpr int C4 = DP / 4;                // float4 per row
  constexpr int PER_T = TR * C4 / NT;       // float4 per thread and tile
  static_assert(TR * C4 % NT == 0 && NG == 4 * G4 + 2 * G2 + G1, "tile");
  static_assert(kFewRows % TR == 0, "tiles fill the padded rows");
  constexpr int XBUF = TR * S;
  constexpr int RED = GRAD ? kFewWaves * kFewTile * DP : 0;
  constexpr int SMF = 2 * XBUF > RED ? 2 * XBUF : RED;
  __shared__ __align__(16) float xs[SMF];
  __shared__ __align__(16) float ys[2][TR];
  __shared__ double lsum[LL ? kFewWaves * kFewTile : 1];

  const int split = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, h = lane >> 4;
  const int64_t n0 = (int64_t)split * a.rows_per_split;
  const int64_t n_end = min(a.N, n0 + a.rows_per_split);
  const int nt = n_end > n0 ? (int)((n_end - n0 + TR - 1) / TR) : 0;

  // resident positions: chunk q, quarter h holds columns 16 q + 4 h .. + 4
  f32x4_t wf[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    wf[q] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    if (l16 < a.C) wf[q] = *(const f32x4_t*)(a.W + l16 * a.ldw + 16 * q + 4 * h);
  }
  f32x4_t g[NG];
#pragma unroll
  for (int k = 0; k < NG; ++k) g[k] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  double lls = 0.0;

  // tile t: TR whole rows of X, one tile in registers ahead of the one in LDS
  // (N_pad is a multiple of kFewRows: the last tile ends inside X and y)
  f32x4_t pre[PER_T];
  float ypre = 0.0f;
  auto load = [&](int t) {
    const f32x4_t* src = (const f32x4_t*)(a.X + (n0 + (int64_t)t * TR) * DP);
#pragma unroll
    for (int k = 0; k < PER_T; ++k) pre[k] = src[tid + k * NT];
    if (tid < TR) ypre = a.y[n0 + (int64_t)t * TR + tid];
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int k = 0; k < PER_T; ++k) {
      const int i = tid + k * NT, row = i / C4, col = i - row * C4;
      *(f32x4_t*)(xs + buf * XBUF + row * S + 4 * col) = pre[k];
    }
    if (tid < TR) ys[buf][tid] = ypre;
  };
  if (nt > 0) {
    load(0);
    store(0);
  }
  __syncthreads();
  for (int t = 0; t < nt; ++t) {
    const int buf = t & 1;
    if (t + 1 < nt) load(t + 1);
    const float* xb = xs + buf * XBUF + wave * 16 * RB * S;
    f32x4_t e[RB];
#pragma unroll
    for (int b = 0; b < RB; ++b) e[b] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      f32x4_t x[RB];
#pragma unroll
      for (int b = 0; b < RB; ++b)
        x[b] = *(const f32x4_t*)(xb + (16 * b + l16) * S + 16 * q + 4 * h);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int b = 0; b < RB; ++b)
          e[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[b][j], wf[q][j], e[b], 0, 0, 0);
    }
    // this lane's rows of the tile: 16 (wave RB + b) + 4 h + v
    const int64_t left = n_end - n0 - (int64_t)t * TR - 16 * RB * wave;
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      const f32x4_t yv = *(const f32x4_t*)(&ys[buf][16 * (wave * RB + b) + 4 * h]);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const bool ok = 16 * b + 4 * h + v < left;
        const float eta = e[b][v];
        if (GRAD) {
          float dll;
          if (LL) {
            double ll;
            glm_both(a.lp, eta, yv[v], dll, ll);
            lls += ok ? ll : 0.0;
          } else {
            dll = glm_dll(a.lp, eta, yv[v]);
          }
          e[b][v] = ok ? dll : 0.0f;
        } else {
          const double ll = a.lp.lik == LIK_BERNOULLI ? -(double)bern_nll_fast(eta, yv[v])
                                                      : glm_ll(a.lp, eta, yv[v]);
          lls += ok ? ll : 0.0;
        }
      }
    }
    if (GRAD) {
#pragma unroll
      for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float* xr = xb + (16 * b + 4 * h + v) * S;
#pragma unroll
          for (int k = 0; k < G4; ++k) {
            const f32x4_t x = *(const f32x4_t*)(xr + 64 * k + 4 * l16);
#pragma unroll
            for (int u = 0; u < 4; ++u)
              g[4 * k + u] =
                  __builtin_amdgcn_mfma_f32_16x16x4f32(e[b][v], x[u], g[4 * k + u], 0, 0, 0);
          }
          if constexpr (G2 != 0) {
            const float2 x = *(const float2*)(xr + 64 * G4 + 2 * l16);
            g[4 * G4] = __builtin_amdgcn_mfma_f32_16x16x4f32(e[b][v], x.x, g[4 * G4], 0, 0, 0);
            g[4 * G4 + 1] =
                __builtin_amdgcn_mfma_f32_16x16x4f32(e[b][v], x.y, g[4 * G4 + 1], 0, 0, 0);
          }
          if constexpr (G1 != 0)
            g[NG - 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                e[b][v], xr[64 * G4 + 32 * G2 + l16], g[NG - 1], 0, 0, 0);
        }
    }
    if (t + 1 < nt) store(buf ^ 1);
    __syncthreads();
  }

  if (GRAD) {
    // element v of accumulator 4 k + u: chain 4 h + v, column 64 k + 4 l16 + u
    // (the 32- and 16-column groups likewise); the waves summed in a fixed
    // order (the tile buffers are not read after the loop's last barrier)
    float* red = xs + wave * kFewTile * DP;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      float* row = red + (4 * h + v) * DP;
#pragma unroll
      for (int k = 0; k < G4; ++k)
        *(f32x4_t*)(row + 64 * k + 4 * l16) =
            f32x4_t{g[4 * k][v], g[4 * k + 1][v], g[4 * k + 2][v], g[4 * k + 3][v]};
      if constexpr (G2 != 0)
        *(float2*)(row + 64 * G4 + 2 * l16) = make_float2(g[4 * G4][v], g[4 * G4 + 1][v]);
      if constexpr (G1 != 0) row[64 * G4 + 32 * G2 + l16] = g[NG - 1][v];
    }
    __syncthreads();
    for (int i = tid; i < a.C * C4; i += NT) {
      f32x4_t s = *(const f32x4_t*)(xs + 4 * i);
#pragma unroll
      for (int w = 1; w < kFewWaves; ++w) s += *(const f32x4_t*)(xs + w * kFewTile * DP + 4 * i);
      *(f32x4_t*)(a.Gpart + ((int64_t)split * a.C + i / C4) * a.ldg + 4 * (i % C4)) = s;
    }
  }
  if (LL) {
    lls += __shfl_xor(lls, 16, 64);
    lls += __shfl_xor(lls, 32, 64);
    if (lane < kFewTile) lsum[wave * kFewTile + lane] = lls;
    __syncthreads();
    if (tid < kFewTile)
      a.llpart[(int64_t)split * a.ll_ld + tid] =
          ((lsum[tid] + lsum[kFewTile + tid]) + lsum[2 * kFewTile + tid]) + lsum[3 * kFewTile + tid];
  }
}

FewPlan few_plan(const edhmc_ctx* ctx, int C);
int few_launch(edhmc_ctx* ctx, const FewArgs& a, int DP, bool grad, bool ll, hipStream_t st);
// X [N_pad][D_pad] -> its first DP columns.
int few_layout(edhmc_ctx* ctx, const float* Xr, int D_pad, int DP, float* Xs, hipStream_t st);

}  // namespace edhmc
