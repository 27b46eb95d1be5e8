// Least squares behind the surrogate's linear skip: the Gram products of a
// sample of the (position, force) pairs, and the solution of the positive
// definite system they make.
#include <algorithm>

#include "common.h"
#include "ctx.h"
#include "../../include/edhmc.h"

namespace edhmc {

typedef __attribute__((ext_vector_type(4))) double f64x4_t;

struct SkipArgs {
  const float *W, *G;
  int64_t P;
  int D;
  const int64_t* idx;
  int n, splits, rows_per;   // rows; splits of them, of rows_per (a multiple of 32)
  const float* nrm;     // in_shift, in_scale, out_shift, out_scale, each Dp
  int Dp;
  int nb, lower;        // 64-column blocks; blocks of the lower triangle
  double *xtx, *xtt;
  double* part;         // [splits][blocks][64][64], or null with one split: straight out
};

// Block t of the products: x^T x's lower triangle first (row by row), then
// x^T t's.
__device__ inline void skip_block(const SkipArgs& a, int t, int& z, int& bi, int& bj) {
  z = t >= a.lower;
  if (z) {
    t -= a.lower;
    bi = t / a.nb;
    bj = t - bi * a.nb;
  } else {
    bi = 0;
    while (t > bi) t -= ++bi;
    bj = t;
  }
}

__device__ inline void skip_store(const SkipArgs& a, int z, int bi, int bj, int i, int j, double v) {
  const int r = bi * 64 + i, c = bj * 64 + j;
  if (r >= a.D || c >= a.D) return;
  (z ? a.xtt : a.xtx)[(int64_t)r * a.D + c] = v;
  if (!z && bi != bj) a.xtx[(int64_t)c * a.D + r] = v;
}

// sum over the rows idx[0..n) of (W, G) of x^T x and x^T t, x = (w - in_shift)
// * in_scale and t = (g - out_shift) / out_scale in fp32, the products and
// sums in FP64 (16x16x4 matrix instructions).  A workgroup makes one 64 x 64
// block over one split of the rows, its four waves 32 x 32 each; 32 rows are
// staged in LDS in fp32 while the next ones come from memory.  An index
// outside [0, P) contributes NaN.
//
// Bound by latency of the gathered rows and the FP64 matrix rate.  n = 32,768,
// D = 512: 128 workgroups of vector FMAs over all the rows 7.6 ms -> 0.65
// (matrix units busy 0.6 of it; loads of one column per thread 0.78).
//
// VEC: 16-byte loads (D a multiple of 4, W and G aligned).
template <bool VEC>
__global__ void __launch_bounds__(256)
skip_gram_kernel(SkipArgs a) {
  constexpr int LD = 80;   // four rows of an operand read in different banks
  __shared__ __align__(16) float la[2][32][LD], lb[2][32][LD];
  int z, bi, bj;
  const int blocks = a.lower + a.nb * a.nb;
  // neighbours in (split, block) order, which read the same rows, on one XCD
  const int at = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const int split = at / blocks, blk = at - split * blocks;
  if (split >= a.splits) return;
  skip_block(a, blk, z, bi, bj);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wi = (wave >> 1) * 32, wj = (wave & 1) * 32, l16 = lane & 15, h = lane >> 4;
  const int r_lo = split * a.rows_per, r_hi = min(a.n, r_lo + a.rows_per);
  // this thread stages columns c .. c + 3 of rows rr and rr + 16
  const int c = (tid & 15) * 4, rr = tid >> 4;
  const int ci = bi * 64 + c, cj = bj * 64 + c;
  const float* Bm = z ? a.G : a.W;
  f32x4_t sh_a, sc_a, sh_b, sc_b;   // columns from D on: anything finite
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int i = min(ci + e, a.D - 1), j = min(cj + e, a.D - 1);
    sh_a[e] = a.nrm[i];
    sc_a[e] = a.nrm[a.Dp + i];
    sh_b[e] = a.nrm[(z ? 2 * a.Dp : 0) + j];
    sc_b[e] = a.nrm[(z ? 3 * a.Dp : a.Dp) + j];
  }
  int64_t src[2];
  f32x4_t va[2], vb[2];
  auto index = [&](int r0) {   // rows past the end: -2
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int row = r0 + rr + 16 * q;
      src[q] = row < r_hi ? a.idx[row] : -2;
      if (row < r_hi && (src[q] < 0 || src[q] >= a.P)) src[q] = -1;
    }
  };
  auto load4 = [&](const float* M, int64_t row, int col) {
    f32x4_t v;
    const float* p = M + max(row, (int64_t)0) * a.D;
    if (VEC) {
      v = *(const f32x4_t*)(p + min(col, a.D - 4));
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = p[min(col + e, a.D - 1)];
    }
    if (row == -1) v = f32x4_t{__builtin_nanf(""), __builtin_nanf(""), __builtin_nanf(""), __builtin_nanf("")};
    return v;
  };
  auto load = [&]() {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      va[q] = load4(a.W, src[q], ci);
      vb[q] = load4(Bm, src[q], cj);
    }
  };
  auto stage = [&](int buf, int r0) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const bool in = r0 + rr + 16 * q < r_hi;
      f32x4_t x, y;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] = (va[q][e] - sh_a[e]) * sc_a[e];
        y[e] = z ? (vb[q][e] - sh_b[e]) / sc_b[e] : (vb[q][e] - sh_b[e]) * sc_b[e];
        x[e] = in ? x[e] : 0.0f;
        y[e] = in ? y[e] : 0.0f;
      }
      *(f32x4_t*)&la[buf][rr + 16 * q][c] = x;
      *(f32x4_t*)&lb[buf][rr + 16 * q][c] = y;
    }
  };
  f64x4_t acc[2][2] = {};
  auto multiply = [&](int buf) {
#pragma unroll
    for (int k = 0; k < 32; k += 4) {
      double x[2], y[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        x[u] = (double)la[buf][k + h][wi + 16 * u + l16];
        y[u] = (double)lb[buf][k + h][wj + 16 * u + l16];
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int v = 0; v < 2; ++v)
          acc[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[u], y[v], acc[u][v], 0, 0, 0);
    }
  };
  if (r_lo < r_hi) {
    index(r_lo);
    load();
    index(r_lo + 32);
    stage(0, r_lo);
    load();
    index(r_lo + 64);
    __syncthreads();
    int buf = 0;
    for (int r0 = r_lo; r0 < r_hi; r0 += 32) {
      multiply(buf);
      stage(buf ^ 1, r0 + 32);
      load();
      index(r0 + 96);
      __syncthreads();
      buf ^= 1;
    }
  }
  // element v of a block: row 4 v + h, column l16
  double* out = a.part + ((int64_t)split * blocks + blk) * 4096;
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = wi + 16 * u + 4 * v + h, j = wj + 16 * w + l16;
        if (a.part) out[i * 64 + j] = acc[u][w][v];
        else skip_store(a, z, bi, bj, i, j, acc[u][w][v]);
      }
}

// Sum of the splits' blocks, in order.
__global__ void __launch_bounds__(256)
skip_sum_kernel(SkipArgs a) {
  const int blocks = a.lower + a.nb * a.nb;
  const int blk = blockIdx.x, e = blockIdx.y * 256 + threadIdx.x;
  const double* p = a.part + (int64_t)blk * 4096 + e;
  double s = 0.0;
#pragma unroll 8
  for (int q = 0; q < a.splits; ++q) s += p[(int64_t)q * blocks * 4096];
  int z, bi, bj;
  skip_block(a, blk, z, bi, bj);
  skip_store(a, z, bi, bj, e >> 6, e & 63, s);
}

// The Gram products; `scratch` (of the engine, kept) holds the splits' blocks.
// Calls on several streams take turns with it: `used` marks the last one's
// end.  Under capture, and where there is no memory for it, one split writes
// straight out.
int skip_gram(edhmc_ctx* ctx, DevBuf& scratch, hipEvent_t& used, const float* W, const float* G,
              int64_t P, int D, const int64_t* idx, int n, const float* nrm, int Dp, double* xtx,
              double* xtt, hipStream_t st) {
  SkipArgs a = {};
  a.W = W; a.G = G; a.P = P; a.D = D; a.idx = idx; a.n = n; a.nrm = nrm; a.Dp = Dp;
  a.nb = (D + 63) / 64;
  a.lower = a.nb * (a.nb + 1) / 2;
  a.xtx = xtx; a.xtt = xtt;
  const int blocks = a.lower + a.nb * a.nb;
  // four workgroups per compute unit, of at least 128 rows
  int splits = std::max(1, std::min(1024 / blocks, (n + 127) / 128));
  a.rows_per = ((n + splits - 1) / splits + 31) / 32 * 32;
  splits = (n + a.rows_per - 1) / a.rows_per;
  if (splits > 1 && !stream_capturing(st) &&
      (used || hipEventCreateWithFlags(&used, hipEventDisableTiming) == hipSuccess) &&
      hipStreamWaitEvent(st, used, 0) == hipSuccess &&
      dev_reserve(ctx, scratch, (size_t)splits * blocks * 4096 * 8) == EDHMC_OK) {
    a.part = (double*)scratch.p;
  } else {
    (void)hipGetLastError();
    splits = 1;
    a.rows_per = (n + 31) / 32 * 32;
  }
  a.splits = splits;
  const dim3 grid((blocks * splits + 7) / 8 * 8);
  if (D % 4 == 0 && ((uintptr_t)W | (uintptr_t)G) % 16 == 0)
    hipLaunchKernelGGL(skip_gram_kernel<true>, grid, dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL(skip_gram_kernel<false>, grid, dim3(256), 0, st, a);
  EDHMC_TRY(check_launch(ctx, "skip_gram"));
  if (!a.part) return EDHMC_OK;
  hipLaunchKernelGGL(skip_sum_kernel, dim3(blocks, 16), dim3(256), 0, st, a);
  EDHMC_TRY(check_launch(ctx, "skip_sum"));
  if (hipEventRecord(used, st) != hipSuccess) return set_err(ctx, EDHMC_EHIP, "skip_gram: event");
  return EDHMC_OK;
}

// One step of a Gauss-Jordan elimination without pivoting of [A | B] (A
// positive definite) by 32 rows: with K the diagonal block of panel k,
// P_j = K^-1 M_kj, row block k becomes P and row block i loses M_ik P.
// Workgroup (j, i) makes block (k + 1 + j, i) of the new matrix from the old
// one (columns up to panel k are not needed again), inverting K for itself.
// After the last panel B's place holds A^-1 B.  A pivot that is not positive
// sets *status.
//
// Bound by the chain of D pivots: 32 of them and two block products a launch,
// 22 us.  D = 512: 0.35 ms, where reading both matrices back and LAPACK's
// general solve took 7.5.
constexpr int kSolveB = 32;

__global__ void __launch_bounds__(256)
solve_step_kernel(const double* __restrict__ M, double* __restrict__ out, int64_t ld, int k,
                  int* __restrict__ status) {
  constexpr int B = kSolveB;
  __shared__ double K[B][B + 1], P[B][B + 1], S[B][B + 1];
  __shared__ double prow[2][B], pcol[2][B];
  const int i = blockIdx.y, j = k + 1 + blockIdx.x;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;   // column; rows ty + 8 u
  double a[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int64_t r = ty + 8 * u;
    a[u] = M[(k * B + r) * ld + k * B + tx];
    P[r][tx] = M[(k * B + r) * ld + j * B + tx];
    S[r][tx] = M[(i * B + r) * ld + k * B + tx];
  }
  // K's inverse in place, a pivot row and column at a time
  bool bad = false;
#pragma unroll
  for (int p = 0; p < B; ++p) {
    if (ty == (p & 7)) prow[p & 1][tx] = a[p >> 3];
    if (tx == p) {
#pragma unroll
      for (int u = 0; u < 4; ++u) pcol[p & 1][ty + 8 * u] = a[u];
    }
    __syncthreads();
    const double piv = prow[p & 1][p], inv = 1.0 / piv;
    bad = bad || !(piv > 0.0);
    const double w = tx == p ? inv : prow[p & 1][tx] * inv;   // the new pivot row
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int r = ty + 8 * u;
      if (r == p) a[u] = w;
      else a[u] = (tx == p ? 0.0 : a[u]) - pcol[p & 1][r] * w;
    }
  }
  if (bad && threadIdx.x == 0) *status = 1;
#pragma unroll
  for (int u = 0; u < 4; ++u) K[ty + 8 * u][tx] = a[u];
  __syncthreads();
  double v[4] = {};
#pragma unroll 8
  for (int q = 0; q < B; ++q) {
    const double b = P[q][tx];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = fma(K[ty + 8 * u][q], b, v[u]);
  }
  double* o = out + (int64_t)i * B * ld + (int64_t)j * B + tx;
  if (i == k) {
#pragma unroll
    for (int u = 0; u < 4; ++u) o[(ty + 8 * u) * ld] = v[u];
    return;
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 4; ++u) P[ty + 8 * u][tx] = v[u];
  __syncthreads();
  double n[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) n[u] = M[((int64_t)i * B + ty + 8 * u) * ld + (int64_t)j * B + tx];
#pragma unroll 8
  for (int q = 0; q < B; ++q) {
    const double b = P[q][tx];
#pragma unroll
    for (int u = 0; u < 4; ++u) n[u] = fma(-S[ty + 8 * u][q], b, n[u]);
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) o[(ty + 8 * u) * ld] = n[u];
}

// M = [A + ridge I | B], both n x n, padded to whole blocks with ones on the
// diagonal.
__global__ void solve_fill_kernel(const double* __restrict__ A, const double* __restrict__ B,
                                  int n, int np, double ridge, double* __restrict__ M,
                                  int* __restrict__ status) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e == 0) *status = 0;
  if (e >= (int64_t)np * 2 * np) return;
  const int i = (int)(e / (2 * np)), c = (int)(e - (int64_t)i * 2 * np);
  const int j = c < np ? c : c - np;
  double v = c < np && i == j ? (i < n ? ridge : 1.0) : 0.0;
  if (i < n && j < n) v += (c < np ? A : B)[(int64_t)i * n + j];
  M[e] = v;
}

// xt[j][i] = X[i][j] in fp32
__global__ void solve_out_kernel(const double* __restrict__ M, int n, int np,
                                 float* __restrict__ xt) {
  __shared__ float t[32][33];
  const int i0 = blockIdx.y * 32, j0 = blockIdx.x * 32, tx = threadIdx.x & 31;
  for (int r = threadIdx.x >> 5; r < 32; r += 8) t[r][tx] = (float)M[(int64_t)(i0 + r) * 2 * np + np + j0 + tx];
  __syncthreads();
  for (int r = threadIdx.x >> 5; r < 32; r += 8)
    if (j0 + r < n && i0 + tx < n) xt[(int64_t)(j0 + r) * n + i0 + tx] = t[tx][r];
}

}  // namespace edhmc

using namespace edhmc;

extern "C" {

int64_t edhmc_solve_spd_work(int32_t n) {
  const int64_t np = ((int64_t)n + kSolveB - 1) / kSolveB * kSolveB;
  return n > 0 ? 2 * np * 2 * np * 8 : 0;
}

int edhmc_solve_spd(edhmc_ctx* ctx, const double* A, const double* B, int32_t n, double ridge,
                    float* xt_out, int32_t* status, void* work, void* stream) {
  if (!ctx) return EDHMC_EINVAL;
  DeviceGuard dg(ctx->device);
  if (!A || !B || !xt_out || !status || !work || n <= 0)
    return set_err(ctx, EDHMC_EINVAL, "bad arguments");
  hipStream_t st = (hipStream_t)stream;
  const int nb = (n + kSolveB - 1) / kSolveB, np = nb * kSolveB;
  const int64_t size = (int64_t)np * 2 * np;
  double* M[2] = {(double*)work, (double*)work + size};
  hipLaunchKernelGGL(solve_fill_kernel, dim3((unsigned)((size + 255) / 256)), dim3(256), 0, st, A,
                     B, n, np, ridge, M[0], status);
  EDHMC_TRY(check_launch(ctx, "solve_fill"));
  for (int k = 0; k < nb; ++k) {
    hipLaunchKernelGGL(solve_step_kernel, dim3(2 * nb - k - 1, nb), dim3(256), 0, st, M[k & 1],
                       M[~k & 1], (int64_t)2 * np, k, status);
    EDHMC_TRY(check_launch(ctx, "solve_step"));
  }
  hipLaunchKernelGGL(solve_out_kernel, dim3(nb, nb), dim3(256), 0, st, M[nb & 1], n, np, xt_out);
  return check_launch(ctx, "solve_out");
}

}  // extern "C"
