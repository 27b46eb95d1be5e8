// Launch side of the one-pass gradient (grad_rows.h).
#include <algorithm>
#include <cmath>

#include "grad_rows.h"

namespace edhmc {

// A row range is addressed with 31-bit byte offsets.
bool rows_ok(const edhmc_ctx* ctx) {
  return ctx->cdt == EDHMC_F32 && ctx->D_pad <= 256 && ctx->D_pad % 64 == 0;
}

// Two workgroups side by side on a compute unit take 10 units, one alone 6
// (measured, both kernels: the other's products fill its waits), and a pair of
// the column-split kernel (32 chains each) takes 0.57 of a chain-split pair (64
// each): the two forms' times over a grid follow from the largest number of
// workgroups on one unit.  us per step, 256 / 384 / 512 / 768 chains, N =
// 100,000, 64 ranges: D = 60 column-split 74 / 108 / 137 / 201, chain-split
// 77 / 127 / 127 / 183; D = 190 177 / 264 / 343 / 574 against 174 / 309 / 312
// / 524.  Where just more than two are due (N = 400,000, D = 190, 1536 chains:
// 576 workgroups) the chain-split one would take 6.1 ms for 4.3.
static int rows_units(int wgs) {
  const int n = (wgs + 255) / 256;
  return 10 * (n / 2) + 6 * (n % 2);
}

bool rows_wide(int C, int splits) {
  return 100 * rows_units((C + 63) / 64 * splits) <= 57 * rows_units((C + 31) / 32 * splits);
}

template <int DP, int CW>
static void launch_cw(RowsArgs a, bool ll, hipStream_t st) {
  a.tiles = (a.C + 16 * CW - 1) / (16 * CW);
  const dim3 grid(a.tiles * a.splits), block(256);
  const bool bern = a.lp.lik == LIK_BERNOULLI;
  if (a.goff && ll) hipLaunchKernelGGL((grad_rows_kernel<DP, CW, true, true, true>), grid, block, 0, st, a);
  else if (a.goff) hipLaunchKernelGGL((grad_rows_kernel<DP, CW, false, true, true>), grid, block, 0, st, a);
  else if (bern && ll) hipLaunchKernelGGL((grad_rows_kernel<DP, CW, true, false, true>), grid, block, 0, st, a);
  else if (bern) hipLaunchKernelGGL((grad_rows_kernel<DP, CW, false, false, true>), grid, block, 0, st, a);
  else if (ll) hipLaunchKernelGGL((grad_rows_kernel<DP, CW, true, false, false>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((grad_rows_kernel<DP, CW, false, false, false>), grid, block, 0, st, a);
}

template <int DP>
static void launch_wide(RowsArgs a, bool ll, hipStream_t st) {
  a.tiles = (a.C + 63) / 64;
  const dim3 grid(a.tiles * a.splits), block(256);
  const bool bern = a.lp.lik == LIK_BERNOULLI;
  if (a.goff && ll) hipLaunchKernelGGL((grad_wide_kernel<DP, true, true, true>), grid, block, 0, st, a);
  else if (a.goff) hipLaunchKernelGGL((grad_wide_kernel<DP, false, true, true>), grid, block, 0, st, a);
  else if (bern && ll) hipLaunchKernelGGL((grad_wide_kernel<DP, true, false, true>), grid, block, 0, st, a);
  else if (bern) hipLaunchKernelGGL((grad_wide_kernel<DP, false, false, true>), grid, block, 0, st, a);
  else if (ll) hipLaunchKernelGGL((grad_wide_kernel<DP, true, false, false>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((grad_wide_kernel<DP, false, false, false>), grid, block, 0, st, a);
}

template <int DP>
static void launch_dp(const RowsArgs& a, bool ll, hipStream_t st) {
  if (a.wide) return launch_wide<DP>(a, ll, st);
  // 16 chains per workgroup while that leaves at most one (64 columns: two) per
  // compute unit.  us per step against 32 chains, N = 100,000, 64 ranges: D =
  // 60, 64 / 128 / 256 chains 32 / 45 / 80 and 47 / 48 / 74; D = 120, 64 / 128
  // chains 48 / 88 and 76 / 78; D = 190 75 / 138 and 103 / 104.  (Of 256 columns
  // three tiles of 64 rows would not fit LDS.)
  if constexpr (DP <= 192) {
    if ((a.C + 15) / 16 * a.splits <= (DP == 64 ? 512 : 256)) return launch_cw<DP, 1>(a, ll, st);
  }
  launch_cw<DP, 2>(a, ll, st);
}

int64_t rows_eta(int C, int splits, int64_t N_pad, bool wide) {
  return wide ? (int64_t)splits * C * kLLTile : N_pad * C;
}

int rows_launch(edhmc_ctx* ctx, RowsArgs a, bool ll, hipStream_t st) {
  if ((a.rows_per_split + 256) * ctx->D_pad * 4 > 0x7fffffffLL)
    return set_err(ctx, EDHMC_EUNSUPPORTED, "one-pass gradient: row range too long");
  switch (ctx->D_pad) {
    case 64: launch_dp<64>(a, ll, st); break;
    case 128: launch_dp<128>(a, ll, st); break;
    case 192: launch_dp<192>(a, ll, st); break;
    case 256: launch_dp<256>(a, ll, st); break;
    default: return set_err(ctx, EDHMC_EUNSUPPORTED, "one-pass gradient: D_pad %d", ctx->D_pad);
  }
  EDHMC_TRY(check_launch(ctx, "grad_rows"));
  if (!ll) return EDHMC_OK;
  const int64_t slots = a.wide ? a.splits + 1 : a.N_pad / kLLTile;
  const dim3 grid((a.C + 7) / 8, (unsigned)std::min<int64_t>(slots, 4096));
  if (a.lp.lik == LIK_BERNOULLI) hipLaunchKernelGGL((rows_ll_kernel<true>), grid, dim3(256), 0, st, a);
  else hipLaunchKernelGGL((rows_ll_kernel<false>), grid, dim3(256), 0, st, a);
  return check_launch(ctx, "rows_ll");
}

__global__ void __launch_bounds__(256)
rows_permute_kernel(const uint32_t* __restrict__ in, int64_t n, uint32_t* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = in[(i & ~15LL) + pi16((int)(i & 15))];
}

int rows_permute(edhmc_ctx* ctx, const void* in, int64_t n, void* out, hipStream_t st) {
  hipLaunchKernelGGL(rows_permute_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                     (const uint32_t*)in, n, (uint32_t*)out);
  return check_launch(ctx, "rows_permute");
}

}  // namespace edhmc
