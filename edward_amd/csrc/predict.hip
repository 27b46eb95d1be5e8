// Launch side of the one-walk posterior predictive (predict.h).
#include <algorithm>

#include "predict.h"

namespace edhmc {

static int predict_q(const edhmc_ctx* ctx) {   // 16-column chunks: any up to 8, then even
  const int q = (ctx->D + 15) / 16;
  return q <= 8 ? q : (q + 1) / 2 * 2;
}

bool predict_ok(const edhmc_ctx* ctx) { return rows_ok(ctx) && ctx->Xp.p; }

PredictPlan predict_plan(const edhmc_ctx* ctx, int S) {
  PredictPlan p;
  constexpr int per = 16 * kPredCB;   // draws per wave
  // four waves along the draws read an X tile once for all of them; fewer
  // where that would compute more than a tenth more draws
  auto pad = [&](int w) { return round_up(S, w * per); };
  // (a tile's two row blocks are work for two waves along the rows)
  p.wc = 10 * pad(4) <= 11 * pad(2) ? 4 : 2;
  p.tiles = (int)(pad(p.wc) / (p.wc * per));
  p.cols = p.tiles * p.wc;
  // as many ranges on every XCD as run together there in one round; where that
  // leaves a fifth of it idle (thousands of draws), up to eight, so that the
  // compute units' shares even out: 5000 draws on 20,000 x 200 762 us with one
  // range on each, 510 with three
  const int slots = predict_q(ctx) <= 8 ? 128 : 64;
  int each = std::max(1, slots / p.tiles);
  if (5 * each * p.tiles < 4 * slots) {
    auto share = [&](int e) { return (e * p.tiles + 31) / 32 / (double)e; };   // of a unit
    for (int e = each + 1; e <= 8; ++e)
      if (share(e) < share(each)) each = e;
  }
  const int64_t want = 8 * each;   // ranges, of at least 128 rows
  p.rows_per_split = std::max<int64_t>(128, round_up((ctx->N + want - 1) / want, 64));
  // a range is addressed with 31-bit byte offsets
  p.rows_per_split = std::min<int64_t>(p.rows_per_split, (0x7fffffffLL / (ctx->D_pad * 4) - 64) / 64 * 64);
  p.splits = (int)((ctx->N + p.rows_per_split - 1) / p.rows_per_split);
  return p;
}

template <int Q>
static void launch_q(const PredictArgs& a, int wc, hipStream_t st) {
  const dim3 grid((a.splits >= 8 ? 8 * ((a.splits + 7) / 8) : a.splits) * a.tiles), block(256);
  const bool bern = a.lp.lik == LIK_BERNOULLI;
  auto go = [&](auto w) {
    constexpr int WC = decltype(w)::value;
    if (bern) hipLaunchKernelGGL((predict_kernel<Q, WC, true>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((predict_kernel<Q, WC, false>), grid, block, 0, st, a);
  };
  if (wc == 4) go(std::integral_constant<int, 4>{});
  else go(std::integral_constant<int, 2>{});
}

int predict_launch(edhmc_ctx* ctx, PredictArgs a, const PredictPlan& p, hipStream_t st) {
  a.tiles = p.tiles;
  a.splits = p.splits;
  a.rows_per_split = p.rows_per_split;
  switch (predict_q(ctx)) {
    case 1: launch_q<1>(a, p.wc, st); break;
    case 2: launch_q<2>(a, p.wc, st); break;
    case 3: launch_q<3>(a, p.wc, st); break;
    case 4: launch_q<4>(a, p.wc, st); break;
    case 5: launch_q<5>(a, p.wc, st); break;
    case 6: launch_q<6>(a, p.wc, st); break;
    case 7: launch_q<7>(a, p.wc, st); break;
    case 8: launch_q<8>(a, p.wc, st); break;
    case 10: launch_q<10>(a, p.wc, st); break;
    case 12: launch_q<12>(a, p.wc, st); break;
    case 14: launch_q<14>(a, p.wc, st); break;
    default: launch_q<16>(a, p.wc, st); break;
  }
  return check_launch(ctx, "predict");
}

}  // namespace edhmc
