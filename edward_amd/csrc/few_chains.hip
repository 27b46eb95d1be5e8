// Launch side of the few-chain gradient (few_chains.h): which calls it takes
// and the split of the rows.
#include <algorithm>
#include <cmath>

#include "few_chains.h"

namespace edhmc {

constexpr int kFewMax = 4;      // chains
constexpr int kCus = 256;
// workgroups per compute unit: three keep enough of X in flight (N = 581,012,
// D = 54, one chain, three transitions of ten steps: 1.86 / 1.38 / 1.26 /
// 1.29 ms with 1 / 2 / 3 / 4), and a fourth only adds partial gradients
constexpr int kFewOcc = 3;

template <typename F>
static bool with_dp(int DP, F f) {
  using std::integral_constant;
  switch (DP) {
    case 16: f(integral_constant<int, 16>{}); return true;
    case 32: f(integral_constant<int, 32>{}); return true;
    case 48: f(integral_constant<int, 48>{}); return true;
    case 64: f(integral_constant<int, 64>{}); return true;
    case 128: f(integral_constant<int, 128>{}); return true;
    case 192: f(integral_constant<int, 192>{}); return true;
    case 256: f(integral_constant<int, 256>{}); return true;
    default: return false;
  }
}

// Up to four chains in fp32 (N = 581,012, D = 54, one chain: 31 us an
// evaluation, 4.7 TB/s of X, against 351 + 236 us for the two-kernel form,
// which pads the chain to 256 and writes and reads 595 MB of residuals;
// N = 1000, D = 10: 4.0 against 15.3 + 5.5 us).  From five chains on the
// two-kernel form's summation order stands: programs of many chains keep
// their bits.
FewPlan few_plan(const edhmc_ctx* ctx, int C) {
  FewPlan p;
  if (ctx->cdt != EDHMC_F32 || ctx->hier || C > kFewMax || ctx->D_pad > 256) return p;
  // columns kept: 16 at a time below 64 (X is all that is read), 64 above
  p.DP = ctx->D <= 48 ? (int)round_up(ctx->D, 16) : ctx->D_pad;
  int occ = 0, rows = 0;
  if (!with_dp(p.DP, [&](auto dp) {
        constexpr int DP = decltype(dp)::value;
        rows = 16 * few_rb(DP) * kFewWaves;
        static const int n = [] {
          int b = 0;
          if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                  &b, few_chains_kernel<DP, true, false>, kFewThreads, 0) != hipSuccess) {
            (void)hipGetLastError();
            b = 0;
          }
          return std::max(1, std::min(b, kFewOcc));
        }();
        occ = n;
      }))
    return p;
  p.on = true;
  // one round of the workgroups that run together, each with at least a tile
  const int64_t row_tiles = (ctx->N + rows - 1) / rows;
  const int64_t s = std::min<int64_t>(kCus * occ, row_tiles);
  p.rows_per_split = (row_tiles + s - 1) / s * rows;
  p.splits = (int)((ctx->N + p.rows_per_split - 1) / p.rows_per_split);
  return p;
}

int few_launch(edhmc_ctx* ctx, const FewArgs& a, int DP, bool grad, bool ll, hipStream_t st) {
  const dim3 grid(a.splits), block(kFewThreads);
  if (!with_dp(DP, [&](auto dp) {
        constexpr int D = decltype(dp)::value;
        if (grad && ll) hipLaunchKernelGGL((few_chains_kernel<D, true, true>), grid, block, 0, st, a);
        else if (grad) hipLaunchKernelGGL((few_chains_kernel<D, true, false>), grid, block, 0, st, a);
        else hipLaunchKernelGGL((few_chains_kernel<D, false, true>), grid, block, 0, st, a);
      }))
    return set_err(ctx, EDHMC_EUNSUPPORTED, "few-chain gradient: %d columns", DP);
  return check_launch(ctx, "few_chains");
}

__global__ void __launch_bounds__(256)
few_layout_kernel(const f32x4_t* __restrict__ Xr, int ld4, int C4, int64_t n4,
                  f32x4_t* __restrict__ Xs) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  const int64_t n = i / C4;
  Xs[i] = Xr[n * ld4 + (i - n * C4)];
}

int few_layout(edhmc_ctx* ctx, const float* Xr, int D_pad, int DP, float* Xs, hipStream_t st) {
  const int64_t n4 = ctx->N_pad * DP / 4;
  hipLaunchKernelGGL(few_layout_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, st,
                     (const f32x4_t*)Xr, D_pad / 4, DP / 4, n4, (f32x4_t*)Xs);
  return check_launch(ctx, "few_layout");
}

}  // namespace edhmc
