// Gradient evaluation in one pass over X for fp32 and D_pad <= 256, any
// number of chains: eta = X W^T, the residuals r(eta, y), G = R^T X, with the
// bits of the two kernels gemm_nt_kernel<float> (GEMM1, GEMM2).
//
// The fp32 matrix instructions are chains of fused multiply-adds in the order
// of their k index (checked on an MI355X against fmaf for 32x32x2 and
// 16x16x4), so a sum keeps its bits as long as its terms keep their order:
//   eta  within every eight columns 0 4 1 5 2 6 3 7 (gemm_nt.h's lane halves);
//   G    the same order of rows, and gemm_nt's row ranges (ksplit).
// Both are had from v_mfma_f32_16x16x4_f32, whose k index is the lane quarter
// h, by one permutation of sixteen: position 4 h + j <-> index
//   pi(4 h + j) = 4 (h & 1) + (h >> 1) + 2 (j & 1) + 8 (j >> 1),
// j counting instructions.  X is kept in a copy with its columns permuted so
// (Xp: a lane's four k of GEMM1 are then 16 contiguous bytes), and lane l of
// GEMM1 takes row pi(l & 15) of a 16-row block: its four results are then
// rows pi(4 h + v), exactly the rows that instruction v of GEMM2 has to
// cover.
//
// Two forms of it, chosen by rows_wide().  grad_rows_kernel: a workgroup of
// four waves owns CT = 16 CW chains and one row range, whose rows it walks in
// order, TR at a time.  Wave (rw, cw) computes the residuals of RB 16-row
// blocks of a tile for chain block cw (positions resident in registers) and
// leaves them in LDS as operand fragments; then every wave multiplies all of
// the tile's fragments by its quarter of X's columns, so that each sum runs
// over the rows in order in one accumulator.  GEMM1 of tile t + 1 and GEMM2 of
// tile t share one phase between two barriers, while tile t + 2 comes from
// memory straight into the third of three LDS buffers (16-byte chunk u of row
// r in slot u ^ (r & 15), so that the operand reads hit disjoint banks).  It
// splits the columns, so that a few chains still make four waves of work.
// grad_wide_kernel, for many chains: below.
//
// Bound: fp32 matrix instructions with many chains (4 N D_pad C operations at
// 155 TF; the bare two products reach 0.83 of it), the serial walk over a
// range's rows with few: one workgroup per range and 16 chains, at most 64
// ranges (their number sets the sums' order).  One evaluation before (two
// GEMMs, the residuals through memory) and here: N = 100,000, D = 256, 1024
// chains 945 -> 804 us; N = 819,200, D = 64, 512 chains with intercepts and
// group sums 1953 -> 1227 us; N = 100,003, D = 101, 50 chains 169 -> 45 us.
#pragma once

#include <type_traits>

#include "common.h"
#include "ctx.h"
#include "gemm_nt.h"

namespace edhmc {

struct RowsArgs {
  const float* Xp;         // [N_pad][DP] row-major, columns in pi order
  const float* yp;         // [N_pad], rows of every 16-row block in pi order
  const float* y;          // [N_pad] in order
  const float* W;          // positions [>= C][DP]
  int64_t N, N_pad;
  int64_t rows_per_split;  // multiple of 16
  int C, tiles, splits;
  bool wide;               // grad_wide_kernel
  LikParams lp;
  float* Gpart;            // [splits][g_ld][DP]
  int64_t g_ld;
  // log-likelihood: FP64 sums over 128 rows llpart [N_pad / 128][ll_ld], and
  // eta [C][128] of the 128-row tiles that rows_ll_kernel sums: in
  // grad_rows_kernel all (eta + tile * C * 128), in grad_wide_kernel those that
  // lie in two row ranges (eta + range where the tile begins * C * 128)
  double* llpart;
  int64_t ll_ld;
  float* eta;
  // hierarchical model: the group intercept goff[c * goff_ld + g] of each
  // row's group g (gidxp in pi order) is added to eta, and the residuals are
  // kept in Rt [N_pad / 16][ldr][16]
  const float* goff;
  int64_t goff_ld;
  const int* gidxp;
  float* Rt;
  int64_t ldr;
  // grad_wide_kernel: group sums ga[c * G + g] of the groups within a row
  // range, group of each row, row offsets of the groups [G + 1]
  float* ga;
  int G;
  const int* gidx;
  const int64_t* off;
};

__host__ __device__ inline int pi16(int p) {
  const int h = p >> 2, j = p & 3;
  return 4 * (h & 1) + (h >> 1) + 2 * (j & 1) + 8 * (j >> 1);
}
__host__ __device__ inline int pi16_inv(int k) {
  return 4 * (((k >> 2) & 1) | ((k & 1) << 1)) + (((k >> 1) & 1) | ((k >> 3) << 1));
}

// The log-likelihood sums its FP64 terms as EpiGLM does (a log ratio of a few
// nats is the difference of two sums of up to a million: it shows the order
// of the sum): the rows of every 64 by a tree over the bits of their index,
// 5 4 3 2 1 0, then the two halves of a 128-row tile.  Summed in the order of
// the walk instead, an evaluation with it was 20 us faster at 50 chains on
// 100,003 x 101 and 80 at 1024 on 100,000 x 256, and log ratios of 0.05 at a
// log joint of a million were off by 1e-9 of themselves.
constexpr int kLLTile = 128;

// 16 bytes per lane from rsrc + off to LDS at dst + 16 lane.
__device__ inline void load_to_lds(__amdgpu_buffer_rsrc_t rsrc, float* dst, int off) {
  typedef __attribute__((address_space(3))) void lds_void;
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void*)dst, 16, off, 0, 0, 0);
}

// a = {low half of a, low half of b}, b = {high half of a, high half of b}
// (halves of the wave's lanes).
__device__ inline void swap_halves(float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, a),
                                                  __builtin_bit_cast(uint32_t, b), false, false);
  a = __builtin_bit_cast(float, (uint32_t)r[0]);
  b = __builtin_bit_cast(float, (uint32_t)r[1]);
}

// Rows 4 h .. 4 h + 3 of a 16-row block, from the lane quarters that hold them
// (element v of quarter h being row pi(4 h + v)).
__device__ inline f32x4_t rows_in_order(const f32x4_t& r) {
  float q0 = r[0], q1 = r[2], q2 = r[1], q3 = r[3];
  swap_halves(q0, q1);
  swap_halves(q2, q3);
  return f32x4_t{q0, q1, q2, q3};
}

// Reads through the scalar unit (p and i uniform over the wave; nothing in the
// kernel writes there).
template <typename T>
__device__ inline T uniform_load(const T* p, int64_t i) {
  typedef const __attribute__((address_space(4))) T* cptr;
  return ((cptr)(uintptr_t)p)[i];
}

// Orders this wave's LDS accesses around it (the hardware does them in order;
// this keeps the compiler from moving them).
__device__ inline void wave_lds_fence() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_wave_barrier();
  asm volatile("" ::: "memory");
}

// Positions of chains c0 .. c0 + 15 (0 from C on) as GEMM1's B operand, lane l
// holding columns 16 q + pi(4 (l >> 4) + j) of chain c0 + (l & 15): read row by
// row and dealt out through 16 DP floats of LDS that are this wave's own (16
// bytes u of row r in slot u ^ r).
template <int DP>
__device__ inline void load_positions(const float* W, int C, int c0, int lane, float* lds,
                                      f32x4_t (&wf)[DP / 16]) {
  constexpr int C4 = DP / 4;
#pragma unroll
  for (int i = 0; i < DP / 16; ++i) {
    const int q = 64 * i + lane, r = q / C4, u = q - r * C4;
    f32x4_t v = {0.0f, 0.0f, 0.0f, 0.0f};
    if (c0 + r < C) v = *(const f32x4_t*)(W + (int64_t)(c0 + r) * DP + 4 * u);
    *(f32x4_t*)(lds + r * DP + 4 * (u ^ r)) = v;
  }
  wave_lds_fence();
  const int l16 = lane & 15, h = lane >> 4;
#pragma unroll
  for (int q = 0; q < DP / 16; ++q)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = 16 * q + pi16(4 * h + j);
      wf[q][j] = lds[l16 * DP + 4 * ((k >> 2) ^ l16) + (k & 3)];
    }
  wave_lds_fence();
}

// 16-row blocks per wave and tile: two where a tile is short otherwise
constexpr int rows_rb(int DP, int CW) { return CW == 2 && DP == 64 ? 2 : 1; }

// BERN: the likelihood (a branch on it would split the unrolled body).
template <int DP, int CW, bool LL, bool HIER, bool BERN>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1)))
grad_rows_kernel(RowsArgs a) {
  static_assert(CW == 1 || CW == 2, "chain blocks per workgroup");
  constexpr int RW = 4 / CW, RB = rows_rb(DP, CW), NB = RB * RW, TR = 16 * NB;
  constexpr int CT = 16 * CW;
  constexpr int Q = DP / 16, NC = DP / 64;   // k chunks of GEMM1; 16-column blocks per wave, GEMM2
  constexpr int C4 = DP / 4;                 // 16-byte chunks per row
  constexpr int LOADS = TR * C4 / 256;       // direct loads per wave and tile (1 KB each)
  static_assert(TR * C4 % 256 == 0, "tile loads");
  constexpr int FR = NB * CW * 256;          // floats of a tile's fragments
  // distinct arrays: a direct load into one does not make reads of another wait
  __shared__ __align__(16) float x0[TR * DP], x1[TR * DP], x2[TR * DP];
  __shared__ __align__(16) float fr[2 * FR];   // fragment (b, cw) of a tile: lane * 4 + v

  int tile, split;
  if (a.splits % 8 == 0) {
    // the chain tiles of one row range run on one XCD and share its L2
    const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
    tile = local % a.tiles;
    split = xcd + 8 * (local / a.tiles);
  } else {
    tile = blockIdx.x % a.tiles;
    split = blockIdx.x / a.tiles;
  }
  LikParams lp = a.lp;
  lp.lik = BERN ? LIK_BERNOULLI : LIK_NORMAL;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cw = wave % CW, rw = wave / CW;
  const int l16 = lane & 15, h = lane >> 4;
  const int c = tile * CT + 16 * cw + l16;       // chain of this lane in GEMM1
  const int64_t n0 = (int64_t)split * a.rows_per_split;
  const int64_t n_end = min(a.N, n0 + a.rows_per_split);
  const int nt = n_end > n0 ? (int)((n_end - n0 + TR - 1) / TR) : 0;

  f32x4_t wf[Q];
  // through 16 rows of a tile buffer that are this wave's own until a tile comes
  load_positions<DP>(a.W, a.C, tile * CT + 16 * cw, lane,
                     (wave < NB ? x0 : x1) + wave % NB * 16 * DP, wf);
  __syncthreads();
  f32x4_t g[CW][NC];
#pragma unroll
  for (int i = 0; i < CW; ++i)
#pragma unroll
    for (int k = 0; k < NC; ++k) g[i][k] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

  // tile t into an X buffer: load i of this wave fills chunks 64 (LOADS wave +
  // i) + lane (rows past the padding: the last row, their residuals are
  // masked)
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(a.Xp + n0 * DP), (short)0, 0x7fffffff, kBufferRsrcWord3);
  int lrow[LOADS], lcol[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int q = 64 * (LOADS * wave + i) + lane;
    lrow[i] = q / C4;
    lcol[i] = ((q - lrow[i] * C4) ^ (lrow[i] & 15)) * 16;
  }
  const int64_t last_row = a.N_pad - 1 - n0;
  auto fetch = [&](int t, float* dst) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int64_t r = min((int64_t)t * TR + lrow[i], last_row);
      load_to_lds(xr, dst + 256 * (LOADS * wave + i), (int)(r * (DP * 4)) + lcol[i]);
    }
  };
  // y (and the groups' intercepts) of this wave's blocks of tile t, loaded a
  // phase before they are used
  f32x4_t yc[RB], oc[RB], yn[RB], on[RB];
  auto rotate = [&]() {
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      yc[b] = yn[b];
      if (HIER) oc[b] = on[b];
    }
  };
  auto rows_of = [&](int t) {
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      const int64_t blk = min(n0 + (int64_t)t * TR + 16 * (rw * RB + b), a.N_pad - 16);
      yn[b] = *(const f32x4_t*)(a.yp + blk + 4 * h);
      if (HIER) {
        const int4 gi = *(const int4*)(a.gidxp + blk + 4 * h);
        const float* o = a.goff + (int64_t)min(c, a.C - 1) * a.goff_ld;
        on[b] = f32x4_t{o[gi.x], o[gi.y], o[gi.z], o[gi.w]};
      }
    }
  };

  const int row_l = pi16(l16);
  const int base1 = (rw * RB * 16 + row_l) * DP;
  const int hx = h ^ row_l;
  // GEMM2: this wave's columns are positions wave DP / 4 + NC l16 + k of the
  // permuted rows
  int off2[4][NC];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int r = pi16(4 * h + v);
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      const int p = wave * (DP / 4) + NC * l16 + k;
      off2[v][k] = r * DP + (((p >> 2) ^ r) << 2) + (p & 3);
    }
  }
  // GEMM1 and residuals of tile t (in X buffer xb) into fragment buffer fb
  auto gemm1 = [&](int t, const float* xb, float* fb) {
    f32x4_t e[RB];
#pragma unroll
    for (int b = 0; b < RB; ++b) e[b] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      f32x4_t x[RB];
#pragma unroll
      for (int b = 0; b < RB; ++b)
        x[b] = *(const f32x4_t*)(xb + base1 + 16 * b * DP + ((hx ^ (4 * q)) << 2));
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int b = 0; b < RB; ++b)
          e[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[b][j], wf[q][j], e[b], 0, 0, 0);
    }
    const int64_t left = n_end - n0 - (int64_t)t * TR;
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      const int blk = rw * RB + b;
      f32x4_t r;
      if (HIER) {
#pragma unroll
        for (int v = 0; v < 4; ++v) e[b][v] = e[b][v] + oc[b][v];
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const bool ok = 16 * blk + pi16(4 * h + v) < left;
        const float eta = e[b][v];
        r[v] = ok ? glm_dll(lp, eta, yc[b][v]) : 0.0f;
      }
      if (LL && 16 * blk < left) {   // not a block of the next range
        const int64_t nb = n0 + (int64_t)t * TR + 16 * blk;
        const f32x4_t o = rows_in_order(e[b]);
        if (c < a.C)
          *(f32x4_t*)(a.eta + ((nb / kLLTile) * a.C + c) * kLLTile + nb % kLLTile + 4 * h) = o;
      }
      *(f32x4_t*)(fb + (blk * CW + cw) * 256 + 4 * lane) = r;
    }
  };
  auto gemm2 = [&](int t, const float* xb, const float* fb) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      f32x4_t r[CW];
#pragma unroll
      for (int i = 0; i < CW; ++i) r[i] = *(const f32x4_t*)(fb + (b * CW + i) * 256 + 4 * lane);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float x[NC];
        if constexpr (NC == 4) {
          const f32x4_t q = *(const f32x4_t*)(xb + 16 * b * DP + off2[v][0]);
          x[0] = q[0]; x[1] = q[1]; x[2] = q[2]; x[3] = q[3];
        } else if constexpr (NC == 2) {
          const float2 q = *(const float2*)(xb + 16 * b * DP + off2[v][0]);
          x[0] = q.x; x[1] = q.y;
        } else {
#pragma unroll
          for (int k = 0; k < NC; ++k) x[k] = xb[16 * b * DP + off2[v][k]];
        }
#pragma unroll
        for (int k = 0; k < NC; ++k)
#pragma unroll
          for (int i = 0; i < CW; ++i)
            g[i][k] = __builtin_amdgcn_mfma_f32_16x16x4f32(r[i][v], x[k], g[i][k], 0, 0, 0);
      }
    }
    if (HIER) {
      // the residuals of the tile, 16 rows of a chain as one 64-byte piece
      const int64_t left = n_end - n0 - (int64_t)t * TR;
      for (int i = tid; i < NB * CT * 4; i += 256) {
        const int part = i & 3, cc = (i >> 2) % CT, b = (i >> 2) / CT;
        const float* f = fb + (b * CW + (cc >> 4)) * 256;
        f32x4_t o;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int p = pi16_inv(4 * part + v);
          o[v] = f[4 * ((p >> 2) * 16 + (cc & 15)) + (p & 3)];
        }
        const int64_t nb = ((n0 + (int64_t)t * TR) >> 4) + b;
        if (16 * b < left)   // not a block of the next range
          *(f32x4_t*)(a.Rt + (nb * a.ldr + tile * CT + cc) * 16 + 4 * part) = o;
      }
    }
  };
  // every load into LDS of this wave done, then everybody's
  auto phase_end = [] {
    __builtin_amdgcn_s_waitcnt(0x0070);   // vmcnt(0) lgkmcnt(0)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  if (nt > 0) {
    fetch(0, x0);
    if (nt > 1) fetch(1, x1);
    rows_of(0);
    rotate();
    rows_of(1);
    phase_end();
    gemm1(0, x0, fr);
    rotate();
    phase_end();
  }
#define EDHMC_ROWS_PHASE(T, XT, XN, XD)                                  \
  if ((T) < nt) {                                                        \
    const int t_ = (T);                                                  \
    if (t_ + 2 < nt) fetch(t_ + 2, XD);                                  \
    rows_of(t_ + 2);                                                     \
    if (t_ + 1 < nt) gemm1(t_ + 1, XN, fr + ((t_ + 1) & 1) * FR);        \
    gemm2(t_, XT, fr + (t_ & 1) * FR);                                   \
    rotate();                                                            \
    phase_end();                                                         \
  }
  for (int t = 0; t < nt; t += 3) {
    EDHMC_ROWS_PHASE(t, x0, x1, x2)
    EDHMC_ROWS_PHASE(t + 1, x1, x2, x0)
    EDHMC_ROWS_PHASE(t + 2, x2, x0, x1)
  }
#undef EDHMC_ROWS_PHASE

  // element v of g[i][k]: chain 16 i + 4 h + v, position p
#pragma unroll
  for (int i = 0; i < CW; ++i)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int cg = tile * CT + 16 * i + 4 * h + v;
      float* row = a.Gpart + ((int64_t)split * a.g_ld + cg) * DP;
#pragma unroll
      for (int k = 0; k < NC; ++k) {
        const int p = wave * (DP / 4) + NC * l16 + k;
        if (cg < a.C) row[(p & ~15) + pi16(p & 15)] = g[i][k][v];
      }
    }
}

// The same gradient for many chains: every wave owns 16 chains with all
// columns of their sums and walks the rows of the range by itself, its
// residuals going from GEMM1 to GEMM2 in registers (the waves share the X
// tiles, with one barrier per tile).  Two workgroups on a compute unit cover
// each other's residual arithmetic and barriers (issuing the next tile's GEMM1
// ahead of this tile's GEMM2 instead costs a third buffer and halves the tile:
// 845 us for 824 with 256 columns, 1290 for 1240 with 64 and group sums).
//
// HIER: sums the residuals per group as it goes, in seg_sum_kernel's order
// (its four lanes per chain are the lane quarters here, rows 4 h .. 4 h + 3
// of every 16-row block), for the groups whose rows lie within the range;
// the residuals of the blocks that other groups reach into go to Rt for that
// kernel.
template <int DP, bool LL, bool HIER, bool BERN>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
grad_wide_kernel(RowsArgs a) {
  constexpr int RB = DP == 64 ? 4 : 2, TR = 16 * RB;   // X tiles of 16 to 32 KB
  constexpr int Q = DP / 16, K4 = DP / 64;
  constexpr int C4 = DP / 4;
  constexpr int LOADS = TR * C4 / 256;
  static_assert(TR * C4 % 256 == 0, "tile loads");
  __shared__ __align__(16) float x0[TR * DP], x1[TR * DP];

  int tile, split;
  if (a.splits % 8 == 0) {
    const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
    tile = local % a.tiles;
    split = xcd + 8 * (local / a.tiles);
  } else {
    tile = blockIdx.x % a.tiles;
    split = blockIdx.x / a.tiles;
  }
  LikParams lp = a.lp;
  lp.lik = BERN ? LIK_BERNOULLI : LIK_NORMAL;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, h = lane >> 4;
  const int c0 = tile * 64 + 16 * wave, c = c0 + l16;
  const int cl = min(c, a.C - 1);
  const int64_t n0 = (int64_t)split * a.rows_per_split;
  const int64_t n_end = min(a.N, n0 + a.rows_per_split);
  const int rows = n_end > n0 ? (int)(n_end - n0) : 0;   // a range's bytes fit 31 bits
  const int nt = (rows + TR - 1) / TR;

  // this wave's own LDS while no tile is in it: 16 rows of a tile buffer
  float* const own = (wave < RB ? x0 : x1) + wave % RB * 16 * DP;
  f32x4_t wf[Q];
  load_positions<DP>(a.W, a.C, c0, lane, own, wf);
  __syncthreads();
  f32x4_t g[Q];
#pragma unroll
  for (int k = 0; k < Q; ++k) g[k] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  double la[4] = {}, lb[4] = {}, first = 0.0;   // even and odd blocks of 64 rows; 64 rows' sum

  int loff[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int q = 64 * (LOADS * wave + i) + lane, r = q / C4;
    loff[i] = (r * C4 + ((q - r * C4) ^ (r & 15))) * 16;
  }
  // tile t into an X buffer (zeros past the padded rows: the tile's resource
  // ends there)
  const int rows_left = (int)min(a.N_pad - n0, (int64_t)1 << 30);
  auto fetch = [&](int t, float* dst) {
    const int r = min(t * TR, rows_left), m = min(TR, rows_left - r);
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.Xp + (n0 + r) * DP), (short)0, m * DP * 4, kBufferRsrcWord3);
#pragma unroll
    for (int i = 0; i < LOADS; ++i) load_to_lds(xr, dst + 256 * (LOADS * wave + i), loff[i]);
  };
  // y of tile t's rows, and the intercepts of their first and last row's
  // groups: loaded at the start of a phase, made ready at its end (rotate), so
  // that no phase ends on a load just issued.  The groups and the row where
  // the first one ends come a phase earlier, through the scalar unit.
  f32x4_t yc[RB], yn[RB], oc[RB];
  float oa[RB], ob[RB];
  int gA[RB], gB[RB];                  // of the tile whose intercepts are loaded
  int eA[RB];                          // its first group's end, rows from n0
  bool two[RB];                        // ... and whether only those two are in the block
  const float* const oc_row = HIER ? a.goff + (int64_t)cl * a.goff_ld : nullptr;
  const int last_blk = rows_left - 16;
  auto rows_of = [&](int t) {
#pragma unroll
    for (int b = 0; b < RB; ++b)
      yn[b] = *(const f32x4_t*)(a.yp + n0 + min(t * TR + 16 * b, last_blk) + 4 * h);
  };
  auto groups_of = [&](int t) {
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      const int64_t n = n0 + min(t * TR + 16 * b, last_blk);
      gA[b] = uniform_load(a.gidx, n);
      gB[b] = uniform_load(a.gidx, n + 15);   // padding: the last group
    }
  };
  auto offsets_of = [&]() {
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      oa[b] = oc_row[gA[b]];
      ob[b] = oc_row[gB[b]];
      const int64_t e = uniform_load(a.off, gA[b] + 1), f = uniform_load(a.off, gB[b]);
      eA[b] = (int)min(e - n0, (int64_t)1 << 30);
      two[b] = f <= e;
    }
  };
  // t: the tile that comes next
  auto rotate = [&](int t) {
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      yc[b] = yn[b];
      if constexpr (HIER) {
        const int n = min(t * TR + 16 * b, last_blk);
        if (gA[b] == gB[b]) {
          oc[b] = f32x4_t{oa[b], oa[b], oa[b], oa[b]};
        } else if (two[b]) {
#pragma unroll
          for (int v = 0; v < 4; ++v) oc[b][v] = n + pi16(4 * h + v) < eA[b] ? oa[b] : ob[b];
        } else {   // three groups or more in 16 rows
          const int4 q = *(const int4*)(a.gidxp + n0 + n + 4 * h);
          oc[b] = f32x4_t{oc_row[q.x], oc_row[q.y], oc_row[q.z], oc_row[q.w]};
        }
      }
    }
  };

  const int row_l = pi16(l16);
  const int hx = h ^ row_l;
  int off2[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int r = pi16(4 * h + v);
    off2[v] = r * DP + ((l16 ^ r) << 2);
  }
  // The scheduling barriers keep the LDS reads two steps ahead of their
  // products: gathered at the front of the unrolled body they would spill.
  auto gemm1 = [&](const float* xb, f32x4_t (&e)[RB]) {
    f32x4_t x[3][RB];
    int sw = hx;
    asm volatile("" : "+v"(sw));   // sixteen addresses kept over the loop would spill
    auto read = [&](int q) {
#pragma unroll
      for (int b = 0; b < RB; ++b)
        x[q % 3][b] = *(const f32x4_t*)(xb + (16 * b + row_l) * DP + ((sw ^ (4 * q)) << 2));
    };
#pragma unroll
    for (int b = 0; b < RB; ++b) e[b] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    read(0);
    read(1);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      if (q + 2 < Q) read(q + 2);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int b = 0; b < RB; ++b)
          e[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[q % 3][b][j], wf[q][j], e[b], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // terms x of a block of rows from nb on (zeros past N) into their 128-row
  // tile's sum
  auto ll_block = [&](int64_t nb, const double (&x)[4]) {
    const int p = (int)(nb >> 4) & 7;
    if (p & 1) {
#pragma unroll
      for (int v = 0; v < 4; ++v) lb[v] += x[v];
    } else {
#pragma unroll
      for (int v = 0; v < 4; ++v) la[v] += x[v];
    }
    const bool last = nb + 16 >= n_end;
    if ((p & 3) != 3 && !last) return;
    double s0 = (la[0] + lb[0]) + (la[2] + lb[2]), s1 = (la[1] + lb[1]) + (la[3] + lb[3]);
    s0 += __shfl_xor(s0, 16, 64);
    s1 += __shfl_xor(s1, 16, 64);
    double s = s0 + s1;
    s += __shfl_xor(s, 32, 64);
#pragma unroll
    for (int v = 0; v < 4; ++v) la[v] = lb[v] = 0.0;
    first = p < 4 ? s : first + s;
    if ((p == 7 || last) && lane < 16 && c < a.C) a.llpart[nb / kLLTile * a.ll_ld + c] = first;
  };
  // residuals of block b of tile t, in place
  auto residual = [&](int t, f32x4_t (&e)[RB], int b) {
    const int64_t nb = n0 + (int64_t)t * TR + 16 * b;
    if (HIER) {
#pragma unroll
      for (int v = 0; v < 4; ++v) e[b][v] = e[b][v] + oc[b][v];
    }
    bool here = false;    // its 128-row tile lies within this range
    if (LL && nb < n_end) {
      const int64_t tb = nb / kLLTile * kLLTile;
      here = tb >= n0 && tb + kLLTile <= n0 + a.rows_per_split;
      if (!here && c < a.C)
        *(f32x4_t*)(a.eta + (tb / a.rows_per_split * a.C + c) * kLLTile + nb % kLLTile + 4 * h) =
            rows_in_order(e[b]);
    }
    double x[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const bool ok = t * TR + 16 * b + pi16(4 * h + v) < rows;
      const float eta = e[b][v];
      float dll;
      if (LL) {
        double ll;
        glm_both(lp, eta, yc[b][v], dll, ll);
        x[v] = ok ? ll : 0.0;
      } else {
        dll = glm_dll(lp, eta, yc[b][v]);
      }
      e[b][v] = ok ? dll : 0.0f;
    }
    if (LL && here) ll_block(nb, x);
  };
  // GEMM2 of a tile
  auto gemm2 = [&](const float* xb, const f32x4_t (&r)[RB]) {
    constexpr int Z = RB * 4 * K4;
    f32x4_t x[3];
    auto read = [&](int z) {
      const int b = z / (4 * K4), v = z / K4 % 4, k = z % K4;
      x[z % 3] = *(const f32x4_t*)(xb + 16 * b * DP + 64 * k + off2[v]);
    };
    read(0);
    read(1);
#pragma unroll
    for (int z = 0; z < Z; ++z) {
      const int b = z / (4 * K4), v = z / K4 % 4, k = z % K4;
      if (z + 2 < Z) read(z + 2);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        g[4 * k + u] = __builtin_amdgcn_mfma_f32_16x16x4f32(r[b][v], x[z % 3][u], g[4 * k + u], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // group of the rows being summed, its last row + 1, and the running sums
  int gc = 0;
  int64_t gend = 0;
  float gsum = 0.0f;
  bool inside = false;
  auto next_group = [&](int64_t n) {   // the group of row n (no empty ones)
    gc = uniform_load(a.gidx, n);
    gend = uniform_load(a.off, gc + 1);
    inside = uniform_load(a.off, gc) >= n0 && gend <= n0 + a.rows_per_split;
    gsum = 0.0f;
  };
  if (HIER && nt > 0) next_group(n0);
  auto segments = [&](int t, const f32x4_t (&r)[RB]) {
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      const int64_t nb = n0 + (int64_t)t * TR + 16 * b;   // first row of the block
      if (nb >= n_end) break;
      const f32x4_t q = rows_in_order(r[b]);
      bool keep = !inside;
      const int64_t be = min(nb + 16, n_end);
      if (gend > be) {   // the block lies within one group that goes on
#pragma unroll
        for (int i = 0; i < 4; ++i) gsum += q[i];
      } else {
        int64_t from = nb;
        while (true) {
          const int64_t to = min(gend, be);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int64_t n = nb + 4 * h + i;
            gsum += (n >= from && n < to) ? q[i] : 0.0f;
          }
          if (gend > be) break;
          if (inside) {
            float s = gsum + __shfl_xor(gsum, 16, 64);
            s += __shfl_xor(s, 32, 64);
            if (h == 0 && c < a.C) a.ga[(int64_t)c * a.G + gc] = s;
          }
          if (gend >= n_end) break;
          from = gend;
          next_group(from);
          keep = keep || !inside;
          if (from >= be) break;
        }
      }
      if (keep) *(f32x4_t*)(a.Rt + ((nb >> 4) * a.ldr + c) * 16 + 4 * h) = q;
    }
  };
  auto phase_end = [] {
    __builtin_amdgcn_s_waitcnt(0x0070);   // vmcnt(0) lgkmcnt(0)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  f32x4_t e[RB];
  if (nt > 0) {
    fetch(0, x0);
    rows_of(0);
    if (HIER) {
      groups_of(0);
      offsets_of();
    }
    rotate(0);
    if (HIER) groups_of(1);
    phase_end();
  }
#define EDHMC_WIDE_PHASE(T, XT, XD)                                      \
  {                                                                      \
    const int t_ = (T);                                                  \
    fetch(t_ + 1, XD);                                                   \
    rows_of(t_ + 1);                                                     \
    if constexpr (HIER) offsets_of();                                    \
    gemm1(XT, e);                                                        \
    _Pragma("unroll") for (int b = 0; b < RB; ++b) residual(t_, e, b);   \
    gemm2(XT, e);                                                        \
    if constexpr (HIER) segments(t_, e);                                 \
    rotate(t_ + 1);                                                      \
    if constexpr (HIER) groups_of(t_ + 2);                               \
    phase_end();                                                         \
  }
  for (int t = 0; t < nt; t += 2) {
    EDHMC_WIDE_PHASE(t, x0, x1)
    EDHMC_WIDE_PHASE(t + 1, x1, x0)
  }
#undef EDHMC_WIDE_PHASE

  // element v of g[4 k + u]: chain c0 + 4 h + v, position 64 k + 4 l16 + u;
  // dealt out through this wave's own LDS, stored row by row
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int r = 4 * h + v;
#pragma unroll
    for (int k = 0; k < Q; ++k) {
      const int p = 64 * (k >> 2) + 4 * l16 + (k & 3), d = (p & ~15) + pi16(p & 15);
      own[r * DP + 4 * ((d >> 2) ^ r) + (d & 3)] = g[k][v];
    }
  }
  wave_lds_fence();
#pragma unroll
  for (int i = 0; i < DP / 16; ++i) {
    const int q = 64 * i + lane, r = q / C4, u = q - r * C4;
    const f32x4_t v = *(const f32x4_t*)(own + r * DP + 4 * (u ^ r));
    if (c0 + r < a.C) *(f32x4_t*)(a.Gpart + ((int64_t)split * a.g_ld + c0 + r) * DP + 4 * u) = v;
  }
}

// The FP64 sums of the tiles whose eta was kept, eight chains per workgroup:
// all tiles, or (wide) one per end of a row range and the tile of padding that
// may come last.
template <bool BERN>
__global__ void __launch_bounds__(256)
rows_ll_kernel(RowsArgs a) {
  const int l = threadIdx.x & 31, c = blockIdx.x * 8 + (threadIdx.x >> 5);
  if (c >= a.C) return;
  LikParams lp = a.lp;
  lp.lik = BERN ? LIK_BERNOULLI : LIK_NORMAL;
  const int64_t tiles = a.N_pad / kLLTile, slots = a.wide ? a.splits + 1 : tiles;
  for (int64_t slot = blockIdx.y; slot < slots; slot += gridDim.y) {
    int64_t tile = slot;
    if (a.wide && slot < a.splits) {
      const int64_t e = (slot + 1) * a.rows_per_split;   // in two ranges, of which this is the first
      tile = e / kLLTile;
      if (e % kLLTile == 0 || tile >= tiles || tile * kLLTile / a.rows_per_split != slot) continue;
    } else if (a.wide) {
      tile = tiles - 1;
      if (tile * kLLTile < a.N) continue;
    }
    const float* eta = a.eta + (slot * a.C + c) * kLLTile;
    double s = 0.0;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      double q = 0.0;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int r = 64 * half + 32 * j + l;
        const int64_t n = tile * kLLTile + r;
        if (n < a.N) {
          float dll;
          double ll;
          glm_both(lp, eta[r], a.y[n], dll, ll);
          q += ll;
        }
      }
#pragma unroll
      for (int off = 16; off > 0; off >>= 1) q += __shfl_xor(q, off, 64);
      s += q;
    }
    if (l == 0) a.llpart[tile * a.ll_ld + c] = s;
  }
}

// Whether the bound data take this kernel (and bind makes Xp and yp).
bool rows_ok(const edhmc_ctx* ctx);
// Whether a call of C chains over this many row ranges is faster with
// grad_wide_kernel (the bits are the same).
bool rows_wide(int C, int splits);
// Floats that RowsArgs.eta holds.
int64_t rows_eta(int C, int splits, int64_t N_pad, bool wide);
// Fills in the chain tiles (C, splits, wide set) and launches.
int rows_launch(edhmc_ctx* ctx, RowsArgs a, bool ll, hipStream_t st);
// out[16 b + p] = in[16 b + pi(p)] for n values (a multiple of 16), 4 bytes each.
int rows_permute(edhmc_ctx* ctx, const void* in, int64_t n, void* out, hipStream_t st);

}  // namespace edhmc
