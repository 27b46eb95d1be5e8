// Whole HMC transitions of a small model in one launch: up to four fp32
// chains, Normal priors, X small enough for the registers of one workgroup.
#pragma once

#include "common.h"
#include "ctx.h"

namespace edhmc {

struct SmallArgs {
  const float* X;          // [N_pad][D_pad]
  const float* y;
  int64_t N;
  int D, D_pad, C, L, T;   // leapfrog steps, transitions
  LikParams lp;
  float lik_weight;
  float half, full;        // fl32(eps / 2), fl32(eps)
  const float* ploc; const float* pscale;
  float* z; float* r; float* g; float* z0; float* g0; float* z_lp;   // [C][D_pad]
  double* logp; double* K0;
  const float* r_fed; const double* u_fed;   // of one transition, or null
  uint64_t seed, counter;                    // counter of the first transition
  float* sample_out;       // [T][C][D] or null
  int32_t* accepted_out; int32_t* n_accept; int32_t* ndiv;
  double* ratio_out;
  double* mom_mean; double* mom_m2; int64_t mom_n;   // draws counted before the first
};

// Whether the context's calls take it.
bool small_ok(const edhmc_ctx* ctx);
int small_launch(edhmc_ctx* ctx, const SmallArgs& a, hipStream_t st);

}  // namespace edhmc
