// Posterior predictive in one walk over X, fp32 with D_pad <= 256: per draw
// the log-likelihood (FP64 sums), per data row the mean response over the
// draws.
//
// A wave owns 16 CB draws, their positions in registers (the other operand of
// v_mfma_f32_16x16x4_f32), and walks 16-row blocks of a row range's X tiles,
// which come straight into LDS.  The result's columns are draws: a lane sums
// its draws' log-likelihood over the rows by itself, and only the mean
// response crosses lanes, summed over the wave's CB blocks first.  X is the
// copy with permuted columns (grad_rows.h), so that eta has the bits of
// gemm_nt_kernel<float>; columns are multiplied 16 at a time, as many as hold
// D.  WC waves of a workgroup take different draws, 4 / WC different rows.
//
// Bound: the matrix instructions (2 N S D operations, D and S rounded up) plus
// exp, log and the FP64 sums: the counters show the matrix cores busy for 350
// K of 645 K cycles and the vector units for 241 K, one after the other
// whatever the waves per SIMD (2 of 64 draws or 4 of 32) or their priorities.
// N = 200,000, D = 100, 500 draws: 320 us, against 477 for
// gemm_nt_kernel with an epilogue that summed every draw over 32 lanes by FP64
// shuffles; D = 10: 165 against 370.
#pragma once

#include "common.h"
#include "ctx.h"
#include "gemm_nt.h"
#include "grad_rows.h"

namespace edhmc {

struct PredictArgs {
  const float* Xp;         // [N_pad][D_pad], columns in pi order
  const float* y;
  const float* W;          // draws [>= S][D_pad]
  int64_t N, N_pad;
  int64_t rows_per_split;  // multiple of 64
  int D_pad, S, tiles, splits;
  LikParams lp;
  double* llpart;          // [splits][ll_ld]
  int64_t ll_ld;
  float* colsum;           // [tiles WC][col_ld] sums over the draws, or null
  int64_t col_ld;
};

constexpr int kPredCB = 2;   // 16-draw blocks per wave

// sum over the 16 lanes of a row of lanes, in all of them
__device__ inline float row16_sum(float v) {
  auto ror = [](float x, auto n) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x120 + decltype(n)::value,
                                           0xf, 0xf, false));
  };
  v += ror(v, std::integral_constant<int, 8>{});
  v += ror(v, std::integral_constant<int, 4>{});
  v += ror(v, std::integral_constant<int, 2>{});
  v += ror(v, std::integral_constant<int, 1>{});
  return v;
}

// Mean response (EpiPredict's) and log-likelihood of one element; glm_ll's
// exponential is the same one.
template <bool BERN>
__device__ inline void predict_terms(const LikParams& lp, float eta, float y, float& mean,
                                     double& ll) {
  ll = glm_ll(lp, eta, y);
  mean = eta;
  if (BERN) {
    const float e = __expf(-fabsf(eta));
    const float inv = fast_rcp(1.0f + e);
    mean = eta >= 0.0f ? inv : e * inv;
  }
}

template <int Q, int WC, bool BERN>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(Q <= 7 ? 4 : Q <= 8 ? 3 : 2)))
predict_kernel(PredictArgs a) {
  constexpr int CB = kPredCB;
  constexpr int RB = 2, TR = 16 * RB;                // row blocks per tile: at most 32 KB
  constexpr int WR = 4 / WC;                         // waves along the rows
  constexpr int C4 = 4 * Q;                          // 16-byte chunks per row
  constexpr int PIECES = TR * C4 / 64;               // direct loads per tile, dealt to the waves
  constexpr int LOADS = (PIECES + 3) / 4;
  static_assert(TR * C4 % 64 == 0 && RB % WR == 0, "tile loads and blocks");
  __shared__ __align__(16) float x0[TR * C4 * 4], x1[TR * C4 * 4];
  // chunk u of row r in slot u ^ swz(r): sixteen rows' chunks hit disjoint banks
  auto swz = [](int r) { return Q % 4 == 0 ? r & 15 : Q % 2 == 0 ? (r >> 1) & 7 : (r >> 2) & 3; };

  // the draws' tiles of one row range run on one XCD and share its L2; fewer
  // ranges than XCDs are spread over all of them
  int tile, split;
  if (a.splits >= 8) {
    const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
    tile = local % a.tiles;
    split = xcd + 8 * (local / a.tiles);
    if (split >= a.splits) return;
  } else {
    tile = blockIdx.x % a.tiles;
    split = blockIdx.x / a.tiles;
  }
  LikParams lp = a.lp;
  lp.lik = BERN ? LIK_BERNOULLI : LIK_NORMAL;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wc = wave % WC, wr = wave / WC;
  const int l16 = lane & 15, h = lane >> 4;
  const int c0 = (tile * WC + wc) * 16 * CB;   // first draw of this wave
  const int64_t n0 = (int64_t)split * a.rows_per_split;
  const int rows = (int)max((int64_t)0, min(a.N - n0, a.rows_per_split));
  const int nt = (rows + TR - 1) / TR;

  // columns 16 q + pi(4 h + j) of draw c0 + 16 b + l16
  f32x4_t wf[CB][Q];
  float dv[CB];   // 1, or 0 for draws from S on (their positions are zeros)
#pragma unroll
  for (int b = 0; b < CB; ++b) {
    const int c = c0 + 16 * b + l16;
    dv[b] = c < a.S ? 1.0f : 0.0f;
    const float* w = a.W + (int64_t)min(c, a.S - 1) * a.D_pad + 4 * (h & 1);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const f32x4_t u = *(const f32x4_t*)(w + 16 * q), v = *(const f32x4_t*)(w + 16 * q + 8);
      const f32x4_t p = h >> 1 ? f32x4_t{u[1], u[3], v[1], v[3]} : f32x4_t{u[0], u[2], v[0], v[2]};
      wf[b][q] = c < a.S ? p : f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }
  double lls[CB];
#pragma unroll
  for (int b = 0; b < CB; ++b) lls[b] = 0.0;

  int loff[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int q = 64 * (4 * i + wave) + lane, r = q / C4;
    loff[i] = r * a.D_pad * 4 + ((q - r * C4) ^ swz(r)) * 16;
  }
  const int rows_left = (int)min(a.N_pad - n0, (int64_t)1 << 30);
  // tile t into an X buffer (zeros past the padded rows)
  auto fetch = [&](int t, float* dst) {
    const int r = min(t * TR, rows_left), m = min(TR, rows_left - r);
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.Xp + (n0 + r) * a.D_pad), (short)0, m * a.D_pad * 4, kBufferRsrcWord3);
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      if (4 * i + wave < PIECES) load_to_lds(xr, dst + 256 * (4 * i + wave), loff[i]);
  };
  const int base = l16 * C4 * 4, hx = h ^ swz(l16);
  auto blocks = [&](int t, const float* xb) {
#pragma unroll
    for (int i = 0; i < RB / WR; ++i) {
      const int k = wr + i * WR;            // block of the tile
      const int r0 = t * TR + 16 * k;       // its first row
      if (r0 >= rows) continue;
      const int64_t nb = n0 + r0;
      const f32x4_t y = *(const f32x4_t*)(a.y + nb + 4 * h);
      f32x4_t e[CB];
#pragma unroll
      for (int b = 0; b < CB; ++b) e[b] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const f32x4_t x = *(const f32x4_t*)(xb + 16 * k * C4 * 4 + base + ((hx ^ (4 * q)) << 2));
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int b = 0; b < CB; ++b)
            e[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[j], wf[b][q][j], e[b], 0, 0, 0);
      }
      // row 4 h + v of the block; rows past the range's end only in its last
      // block (a branch per block instead of a mask per element)
      f32x4_t s = {0.0f, 0.0f, 0.0f, 0.0f};
      auto terms = [&](auto ragged) {
#pragma unroll
        for (int b = 0; b < CB; ++b)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            float mean;
            double ll;
            predict_terms<BERN>(lp, e[b][v], y[v], mean, ll);
            if (decltype(ragged)::value) ll = r0 + 4 * h + v < rows ? ll : 0.0;
            lls[b] += ll;
            s[v] = fmaf(mean, dv[b], s[v]);
          }
      };
      if (r0 + 16 <= rows) terms(std::false_type{});
      else terms(std::true_type{});
      if (a.colsum) {
#pragma unroll
        for (int v = 0; v < 4; ++v) s[v] = row16_sum(s[v]);
        if (l16 == 0)   // whole blocks: col_ld >= N_pad
          *(f32x4_t*)(a.colsum + (int64_t)(tile * WC + wc) * a.col_ld + nb + 4 * h) = s;
      }
    }
  };
  auto phase_end = [] {
    __builtin_amdgcn_s_waitcnt(0x0070);   // vmcnt(0) lgkmcnt(0)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  if (nt > 0) fetch(0, x0);
  phase_end();
  for (int t = 0; t < nt; t += 2) {
    if (t + 1 < nt) fetch(t + 1, x1);
    blocks(t, x0);
    phase_end();
    if (t + 1 < nt) {
      if (t + 2 < nt) fetch(t + 2, x0);
      blocks(t + 1, x1);
      phase_end();
    }
  }
  // over the lane quarters, then over the waves along the rows
  double* sm = (double*)x0;   // [WR][WC][CB][16]
#pragma unroll
  for (int b = 0; b < CB; ++b) {
    double s = lls[b];
    s += __shfl_xor(s, 16, 64);
    s += __shfl_xor(s, 32, 64);
    if (lane < 16) sm[((wr * WC + wc) * CB + b) * 16 + lane] = s;
  }
  __syncthreads();
  for (int i = tid; i < WC * CB * 16; i += 256) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < WR; ++w) s += sm[w * WC * CB * 16 + i];
    const int c = tile * WC * CB * 16 + i;
    if (c < a.S) a.llpart[(int64_t)split * a.ll_ld + c] = s;
  }
}

// Whether the bound data take this kernel.
bool predict_ok(const edhmc_ctx* ctx);
// wc: waves along the draws; cols: partial sums over the draws per row.
struct PredictPlan {
  int wc, tiles, splits, cols;
  int64_t rows_per_split;
};
PredictPlan predict_plan(const edhmc_ctx* ctx, int S);
int predict_launch(edhmc_ctx* ctx, PredictArgs a, const PredictPlan& p, hipStream_t st);

}  // namespace edhmc
