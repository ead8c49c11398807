// mcr_device.hip -- gfx950 kernels of the Monte Carlo crash-risk model.
//
// Replaces monte_carlo_kernel (src/05-GPU/monte_carlos_cuda.cu:23-72) and the host
// Cholesky it relies on (:84-93).  Per path p the reference computes
//   Z ~ N(0, I_N), R = mu + L Z (lower-triangular, :51-57), S = #{R_i < -x} (:60-65),
//   extreme iff S >= k (:69-71), and stores S (:67).
// Here:
//   k_chol_step  FP64 Cholesky and the portfolio loading v = L^T w, one launch per
//                32 columns, many workgroups.
//   k_factor     one workgroup behind them: w^T mu and ||v||, the query's record, and
//                the jitter policy's retries where the first attempt failed.
//   k_prep       fp32 / bf16 layouts of the factor for the path kernels.
//   k_collect    the query's results to pinned host memory.
//   k_valu_reg   fused path kernel, one path per lane, n <= 64 rows in registers,
//                factor read through the scalar cache: r_i = mu_i then fmaf(L_ij, z_j)
//                for j = 0..i, exactly the order the C mirror uses.
//   k_wave       fp32, 64 < n <= 127: 64 paths per wave on v_mfma_f32_32x32x2_f32,
//                whose row sums are the same fmaf chains.
//   k_f32_lds    fp32, n <= 1024: 64 paths per workgroup, their normals staged in
//                LDS as operands of the same instruction.
//   k_mfma       32 paths per wave on v_mfma_f32_32x32x16_bf16: A = factor rows
//                (bf16 hi/lo), B = normals (bf16 hi/lo), three products per step
//                (hi*hi + hi*lo + lo*hi), fp32 accumulation, n <= 127.
//   k_mfma_stage the same products, n = 128-511: 64 paths per workgroup, all their
//                normals staged in LDS before they are multiplied.
//   k_mfma_spec  the same, n = 512-767: waves that multiply beside waves that generate.
// Every path kernel reduces the exceedance count, tail counts and fixed-point
// tail sums in registers (k_valu_reg, k_mfma_spec) or LDS and adds them to the
// query's with one atomic per workgroup and counter; no normal ever leaves the
// chip.
#include <mutex>

#include "mcr_kern_common.h"

namespace mcr {

// ---------------------------------------------------------------------------
// Factor: FP64 Cholesky of A + delta I, then the portfolio moments.
// Jitter policy: delta_0 = 0, delta_t = mean(diag) 10^(t-12) for t = 1..8, then
// the modified factorisation with failing pivots clamped to delta_8.  A pivot
// fails when it is not above n eps (A_jj + delta).
// The first attempt runs on many workgroups, one launch per 32 columns
// (k_chol_step); the rare retries, and the report of non-finite input, are the
// finishing kernel's, on one workgroup (cholesky_body), with the same arithmetic
// in the same order.
// ---------------------------------------------------------------------------
__device__ double block_sum_f64(double v, double* red) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  v = wave_sum_f64(v);
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  double s = 0.0;
  const int nw = (blockDim.x + 63) >> 6;
  for (int i = 0; i < nw; ++i) s += red[i];
  return s;
}

// Retries (attempts 2 to 10) of a factorisation whose first attempt failed, or
// the rejection of non-finite input.
// FP64 Cholesky of A + delta I into L (row-major, zero upper triangle) on one
// workgroup of 1024 threads, right-looking by panels of kPanel columns:
//   panel:    thread r holds row k0 + r of the panel in registers; column c is
//             finished with one barrier: rows c..kb-1 publish their column-c
//             entry (double-buffered LDS slot), every row tests the same
//             pivot, scales its entry and updates its later panel columns;
//   trailing: A22 -= L21 L21^T on the lower triangle, 4 x 4 register tiles
//             read from a column-major LDS copy of the panel.
// Jitter policy: try t = 1..9 adds delta_t = mean(diag A) * 10^(min(t,8)-12);
// try 9 clamps failing pivots to delta.  A pivot fails when it
// is not above n eps (A_jj + delta).  Returns false (and records attempts =
// -1) for non-finite A.
constexpr int kPanel = 16;
// MAXN: the largest n the kernel is built for (kMaxN: 78 KiB of LDS; the
// column-chunk queries' kChunkMaxN: 129 KiB); a panel row per thread.
template <int MAXN>
struct FactorShared {
  static constexpr int kLd = (MAXN + 3) / 4 * 4 + 4;  // rows + tile overrun, multiple of 4
  __attribute__((aligned(16))) double panel[kPanel * kLd];  // [c * kLd + r]
  double pivot[2][kPanel];
  double adiag[kPanel];  // A_jj + delta of the panel's columns (pivot tolerance)
  double red[16];
};

template <int MAXN>
__device__ bool cholesky_body(const FactorArgs& a, FactorShared<MAXN>& sh, int* attempts_out,
                              int* clamped_out, int* fail_out, double* delta_out) {
  const int n = a.n;
  const int tid = threadIdx.x, nthr = blockDim.x;  // nthr >= MAXN: every panel row has an owner
  constexpr int kPanelLd = FactorShared<MAXN>::kLd;
  const int lane = tid & 63, wave = tid >> 6, nwave = nthr >> 6;
  const double* __restrict__ A = a.A;
  double* __restrict__ L = a.L;

  double bad = 0.0, dsum = 0.0;
  for (int e = tid; e < n * n; e += nthr)
    if (!isfinite(A[e])) bad = 1.0;
  if (tid < n) dsum = A[tid * n + tid];
  bad = block_sum_f64(bad, sh.red);
  dsum = block_sum_f64(dsum, sh.red);
  if (bad > 0.0) {
    if (tid == 0) {
      a.info->attempts = -1;
      a.info->clamped = 0;
      a.info->fail_col = 0;
      a.info->jitter = 0.0;
      if (a.finfo) *a.finfo = *a.info;
    }
    return false;
  }
  const double mean = dsum / (double)n;

  int attempts = 0, clamped = 0, fail = 0, last_fail = 0;
  double delta = 0.0;
  for (int t = 1; t <= 9; ++t) {
    const bool clamp = (t == 9);
    delta = mean * pow(10.0, (double)((t < 8 ? t : 8) - 12));
    fail = 0;
    clamped = 0;
    for (int i = wave; i < n; i += nwave)
      for (int j = lane; j < n; j += 64) {
        const size_t e = (size_t)i * n + j;
        L[e] = (j < i) ? A[e] : (j == i ? A[e] + delta : 0.0);
      }
    __syncthreads();

    for (int k0 = 0; k0 < n && !fail; k0 += kPanel) {
      const int kb = min(kPanel, n - k0), rows = n - k0;
      const int r = tid;
      const bool own = r < rows;
      double x[kPanel];
#pragma unroll
      for (int c = 0; c < kPanel; ++c)
        x[c] = (own && c < kb) ? L[(size_t)(k0 + r) * n + k0 + c] : 0.0;
      if (tid < kb) sh.adiag[tid] = A[(size_t)(k0 + tid) * n + k0 + tid] + delta;

#pragma unroll
      for (int c = 0; c < kPanel; ++c) {
        const bool live = c < kb && !fail;  // uniform over the workgroup
        if (live && own && r >= c && r < kb) sh.pivot[c & 1][r] = x[c];
        __syncthreads();
        if (live) {
          const int j = k0 + c;
          double d = sh.pivot[c & 1][c];
          const double tol = (double)n * DBL_EPSILON * sh.adiag[c];
          if (!(d > tol) || !isfinite(d)) {
            if (clamp && isfinite(d)) {
              d = delta;
              ++clamped;
            } else {
              fail = j + 1;
            }
          }
          if (!fail) {
            const double ljj = sqrt(d);
            const double rl = 1.0 / ljj;
            if (own && r == c) x[c] = ljj;
            if (own && r > c) {
              const double lr = x[c] * rl;
              x[c] = lr;
#pragma unroll
              for (int c2 = c + 1; c2 < kPanel; ++c2)
                if (c2 < kb && r >= c2) x[c2] = fma(-lr, sh.pivot[c & 1][c2] * rl, x[c2]);
            }
          }
        }
      }
      if (fail) break;

      if (own) {
#pragma unroll
        for (int c = 0; c < kPanel; ++c) {
          if (c < kb) L[(size_t)(k0 + r) * n + k0 + c] = x[c];
          sh.panel[c * kPanelLd + r] = x[c];
        }
      }
      for (int e = tid; e < kPanel * (kPanelLd - rows); e += nthr) {
        const int c = e / (kPanelLd - rows), q = e % (kPanelLd - rows);
        sh.panel[c * kPanelLd + rows + q] = 0.0;
      }
      __syncthreads();

      // trailing update of columns k1..n-1 (only when the panel was full)
      const int k1 = k0 + kb, m = n - k1;
      if (m > 0) {
        const int TB = (m + 3) >> 2;
        const int ntiles = TB * (TB + 1) / 2;
        for (int tt = tid; tt < ntiles; tt += nthr) {
          int bi = (int)((sqrt(8.0 * tt + 1.0) - 1.0) * 0.5);
          while (bi * (bi + 1) / 2 > tt) --bi;
          while ((bi + 1) * (bi + 2) / 2 <= tt) ++bi;
          const int bj = tt - bi * (bi + 1) / 2;
          const int ri = kPanel + 4 * bi, rj = kPanel + 4 * bj;
          double acc[4][4];
#pragma unroll
          for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[u][v] = 0.0;
#pragma unroll 1
          for (int p = 0; p < kPanel; ++p) {
            const double2* pa = (const double2*)&sh.panel[p * kPanelLd + ri];
            const double2* pb = (const double2*)&sh.panel[p * kPanelLd + rj];
            const double2 a01 = pa[0], a23 = pa[1], b01 = pb[0], b23 = pb[1];
            const double av[4] = {a01.x, a01.y, a23.x, a23.y};
            const double bv[4] = {b01.x, b01.y, b23.x, b23.y};
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
              for (int v = 0; v < 4; ++v) acc[u][v] = fma(av[u], bv[v], acc[u][v]);
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int i = k1 + 4 * bi + u;
            if (i >= n) break;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
              const int j = k1 + 4 * bj + v;
              if (j <= i) L[(size_t)i * n + j] -= acc[u][v];
            }
          }
        }
      }
      __syncthreads();
    }
    attempts = t + 1;
    last_fail = fail;
    if (!fail) break;
  }
  *attempts_out = attempts;
  *clamped_out = clamped;
  *fail_out = last_fail;
  *delta_out = delta;
  return true;
}

// v_j = sum_{i >= j} L_ij w_i, i ascending; the loads of 32 rows are in flight
// together (one at a time cost a memory latency per row).
__device__ __forceinline__ double loading_of(const FactorArgs& a, int j) {
  const int n = a.n;
  const double* __restrict__ col = a.L + j;
  double s = 0.0;
  int i = j;
  for (; i + 32 <= n; i += 32) {
    double l[32];
#pragma unroll
    for (int u = 0; u < 32; ++u) l[u] = col[(size_t)(i + u) * n];
#pragma unroll
    for (int u = 0; u < 32; ++u) s += l[u] * a.w[i + u];
  }
  for (; i < n; ++i) s += col[(size_t)i * n] * a.w[i];
  return s;
}

// Portfolio loading v = L^T w, mean w^T mu and sd ||v|| in FP64, and the
// query's record (factor outcome, moments, VaR windows).
// The columns before j0 have their v_j already.
__device__ void moments_body(const FactorArgs& a, double* red, int j0, int attempts, int clamped,
                             int last_fail, double delta) {
  const int n = a.n;
  const int tid = threadIdx.x;
  __syncthreads();
  for (int j = j0 + tid; j < n; j += blockDim.x) a.v64[j] = loading_of(a, j);
  __syncthreads();
  double mp = 0.0, ss = 0.0;
  for (int i = tid; i < n; i += blockDim.x) {
    mp += a.w[i] * a.mu[i];
    ss += a.v64[i] * a.v64[i];
  }
  mp = block_sum_f64(mp, red);
  ss = block_sum_f64(ss, red);
  if (tid == 0) {
    DevInfo* info = a.info;
    info->attempts = attempts;
    info->clamped = clamped;
    info->fail_col = last_fail;
    info->jitter = delta;
    info->mp = mp;
    const double sd = sqrt(ss);
    info->loss_sd = sd;
    for (int al = 0; al < kMaxAlpha; ++al) {
      if (al < a.n_alpha) {
        info->lo[al] = (float)(-mp + (a.za[al] - a.ha[al]) * sd);
        info->hi[al] = (float)(-mp + (a.za[al] + a.ha[al]) * sd);
      } else {
        info->lo[al] = 0.0f;
        info->hi[al] = 0.0f;
      }
    }
    info->hist_lo = 0.0f;
    info->hist_scale = 0.0f;
  }
}


// ---------------------------------------------------------------------------
// First attempt, launch s of ceil(n / 32): block column s (columns 32s .. 32s +
// 31) is finished and the columns right of it take the update of block column
// s - 1, which only needs what launch s - 1 left behind:
//   panels        a workgroup per 32 rows below the diagonal block, which each
//                 factors for itself: 64 rows come in coalesced and take block
//                 column s - 1's update on v_mfma_f64_16x16x4, then 16 columns
//                 at a time go through the first wave, a row per lane, the
//                 pivots and the diagonal block's entries coming by readlane.
//   update tiles  64 x 64, block column s - 1's product subtracted (same
//                 instruction);
//   loading       pieces of v = L^T w, a column per lane (see chol_loading).
// Every entry sees the operations of a right-looking factorisation by panels of
// 16 columns in its order (per panel a chain of 16 fused multiply-adds from zero,
// then one subtraction; inside a panel one fused multiply-add per column), so L
// has the bits that cholesky_body's algorithm gives it.
// Bound: the chain of 32 square roots and reciprocals of a launch (3.7 of its 10
// us at n = 600), then the latency of its loads.  All launches, n = 15 / 143 /
// 301 / 600 / 1024: 13 / 47 / 92 / 178 / 313 us; with a row per lane in global
// memory too (64 lines to a load) and the update on the vector unit, its operands
// broadcast from LDS, 20 / 114 / 251 / 413 / 775; on one workgroup 1809 us at n =
// 600, 6768 at n = 1024.
// ---------------------------------------------------------------------------
constexpr int kBlk = 32;
constexpr int kLoadRows = 128;  // rows of L^T w in LDS at a time

// double of lane `src` (a constant) in every lane
__device__ __forceinline__ double bcast(double v, int src) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)b, src);
  const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(b >> 32), src);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

typedef double f64x4 __attribute__((ext_vector_type(4)));

struct CholShared {
  union {
    struct {
      double prev[64][33];  // block column s - 1 in the panel's rows
      double x[64][34];     // block column s there
    } p;
    struct {
      double a[64][33], b[64][33];  // block column s - 1 in the tile's rows and columns
    } u;
    double prod[kLoadRows][kBlk];  // L_ij w_i
  };
  int failed;
} __attribute__((aligned(16)));

// 16 x 16 products of rows ra .. and rb .. over 16 columns from p: a chain of 16
// fused multiply-adds from zero per entry, p ascending (the instruction fuses
// and takes its four products in that order).  Entry i of lane l: row
// 4 i + l / 16, column l % 16.
template <int LD>
__device__ __forceinline__ f64x4 chain16(const double (&va)[64][LD], int ra,
                                         const double (&vb)[64][LD], int rb, int p) {
  const int lane = threadIdx.x & 63, m = lane & 15, k = lane >> 4;
  f64x4 acc = {};
#pragma unroll
  for (int q = 0; q < 16; q += 4)
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(va[ra + m][p + q + k], vb[rb + m][p + q + k], acc, 0, 0, 0);
  return acc;
}

// sqrt(d) and its correctly rounded reciprocal in kStages steps (all with one
// use of the vector unit's latency), without the library's care for the ends of
// the range: d in [2^-752, 2^1000].  Goldschmidt's coupled iteration for the
// root and half its reciprocal from the hardware's estimate, then Markstein's
// correction of each by its fused residual ("Computation of elementary functions
// on the IBM RISC System/6000 processor", 1990); the reciprocal starts from the
// root's instead of an estimate of its own.  The same bits as sqrt(d) and 1.0 /
// sqrt(d) over 2e8 random, square and near-square d, except where the root's
// significand is all ones (below): there the corrected reciprocal is a tie that
// rounds to even, one unit in the last place low.
struct RootRecip {
  double d, g, h, q, e;
  static constexpr int kStages = 10;
  __device__ __forceinline__ void stage(int k) {
    if (k == 0) h = __builtin_amdgcn_rsq(d);
    if (k == 1) g = d * h, h = 0.5 * h;
    if (k == 2) e = fma(-h, g, 0.5);
    if (k == 3) g = fma(g, e, g), h = fma(h, e, h);
    if (k == 4) e = fma(-g, g, d), q = h + h;
    if (k == 5) g = fma(e, h, g);
    if (k == 6) e = fma(-g, g, d), d = fma(-g, q, 1.0);
    if (k == 7) g = fma(e, h, g), q = fma(d, q, q);
    if (k == 8) e = fma(-g, q, 1.0);
    if (k == 9) q = fma(e, q, q);
  }
};

// d is one of the last two doubles below a power of four, whose root rounds to
// the last double below a power of two.
__device__ __forceinline__ bool root_all_ones(double d) {
  return (__builtin_bit_cast(uint64_t, d) & 0x001ffffffffffffeull) == 0x000ffffffffffffeull;
}

// Columns q .. q + 15 of the panel, a row per lane (rows 0-31 the diagonal
// block's): x the row's entries, piv the pivot of the lane's column as found.
// Not for columns with a root_all_ones pivot.
// One wave runs this alone, so instruction order is what hides latency: the next
// column takes its update first, and a step of its root stands before each of
// the other columns' updates.  All launches, n = 143 / 301 / 600: 47 / 92 / 194
// us; a column after the other 50 / 98 / 201, with the library's root and
// reciprocal 55 / 107 / 213.
__device__ __forceinline__ void chol_columns(double (&x)[kPanel], int q, double* piv) {
  const int lane = threadIdx.x & 63;
  RootRecip rt;
  rt.d = bcast(x[0], q);
  if (lane == q) *piv = rt.d;
#pragma unroll
  for (int k = 0; k < RootRecip::kStages; ++k) rt.stage(k);
#pragma unroll
  for (int c = 0; c < kPanel; ++c) {
    const double lr = x[c] * rt.q;
    x[c] = lane == q + c ? rt.g : lr;
    if (c + 1 == kPanel) break;
    x[c + 1] = fma(-lr, bcast(lr, q + c + 1), x[c + 1]);
    rt.d = bcast(x[c + 1], q + c + 1);
    if (lane == q + c + 1) *piv = rt.d;
#pragma unroll
    for (int k = 0; k < RootRecip::kStages; ++k) {
      rt.stage(k);
      const int c2 = c + 2 + k;
      if (c2 < kPanel) x[c2] = fma(-lr, bcast(lr, q + c2), x[c2]);
    }
#pragma unroll
    for (int c2 = c + 2 + RootRecip::kStages; c2 < kPanel; ++c2) x[c2] = fma(-lr, bcast(lr, q + c2), x[c2]);
  }
}

// The same with the library's root and reciprocal, for pivots of any size.
__device__ __forceinline__ void chol_columns_any(double (&x)[kPanel], int q, double* piv) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int c = 0; c < kPanel; ++c) {
    const double d = bcast(x[c], q + c);
    if (lane == q + c) *piv = d;
    const double ljj = sqrt(d), rl = 1.0 / ljj;
    const double lr = x[c] * rl;
    x[c] = lane == q + c ? ljj : lr;
#pragma unroll
    for (int c2 = c + 1; c2 < kPanel; ++c2) x[c2] = fma(-lr, bcast(lr, q + c2), x[c2]);
  }
}

__device__ void chol_panel(const FactorArgs& a, int s, int blk, CholShared& sh) {
  const int n = a.n, k0 = kBlk * s, kb = min(kBlk, n - k0);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double* __restrict__ L = a.L;
  // row t of the panel: the diagonal block's, then the workgroup's own
  auto row_of = [&](int t) { return t < kBlk ? k0 + t : k0 + kBlk * blk + t; };

  // entry i of half h: row 16 wave + 4 i + lane / 16, column 16 h + lane % 16
  f64x4 x[2];
  const bool diag = wave < 2;
  // the diagonal block, which one workgroup finishes while others may still have
  // to read it, waits in the zero triangle (see chol_update)
  const double* __restrict__ src = s <= 1 ? a.A : diag ? L - (size_t)kBlk * n : L;
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = 16 * wave + 4 * i + (lane >> 4), c = 16 * h + (lane & 15), row = row_of(t);
      x[h][i] = row < n && c < kb && (!diag || c <= t) ? src[(size_t)row * n + k0 + c]
                                                       : (diag && c == t ? 1.0 : 0.0);  // identity pads
    }
  if (s > 0) {
    double l[64 * kBlk / 256];
#pragma unroll
    for (int u = 0; u < 64 * kBlk / 256; ++u) {
      const int t = 8 * u + threadIdx.x / kBlk, row = row_of(t);
      l[u] = row < n ? L[(size_t)row * n + k0 - kBlk + threadIdx.x % kBlk] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < 64 * kBlk / 256; ++u)
      sh.p.prev[8 * u + threadIdx.x / kBlk][threadIdx.x % kBlk] = l[u];
    __syncthreads();
#pragma unroll
    for (int p = 0; p < kBlk; p += kPanel)
#pragma unroll
      for (int h = 0; h < 2; ++h) x[h] -= chain16(sh.p.prev, 16 * wave, sh.p.prev, 16 * h, p);
  }
  // the block's diagonal of A: its pivots are no larger, and none is smaller than
  // n eps of its own but one that fails
  const bool col = lane < kb;
  const double ajj = col ? a.A[(size_t)(k0 + lane) * n + k0 + lane] : 1.0;
  const bool mid = __ballot(!(ajj > 0x1p-700 && ajj < 0x1p+990)) == 0ull;
  // 16 columns at a time: into LDS, through the first wave's registers and back
  double piv = 0.0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (kPanel * h >= kb) break;
    if (h > 0) x[h] -= chain16(sh.p.x, 16 * wave, sh.p.x, kPanel, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      sh.p.x[16 * wave + 4 * i + (lane >> 4)][kPanel * h + (lane & 15)] = x[h][i];
    __syncthreads();
    if (wave == 0) {
      double y[kPanel];
      bool any = !mid;
      if (mid) {
#pragma unroll
        for (int c = 0; c < kPanel; ++c) y[c] = sh.p.x[lane][kPanel * h + c];
        chol_columns(y, kPanel * h, &piv);
        // the first such pivot is right, as the columns before it are
        any = __ballot(root_all_ones(piv)) != 0ull;
      }
      if (any) {
#pragma unroll
        for (int c = 0; c < kPanel; ++c) y[c] = sh.p.x[lane][kPanel * h + c];
        chol_columns_any(y, kPanel * h, &piv);
      }
#pragma unroll
      for (int c = 0; c < kPanel; ++c) sh.p.x[lane][kPanel * h + c] = y[c];
    }
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < 64 * kBlk / 256; ++u) {
    const int t = 8 * u + threadIdx.x / kBlk, c = threadIdx.x % kBlk, row = row_of(t);
    if (row < n && c < kb && (t >= kBlk || blk == 0))
      L[(size_t)row * n + k0 + c] = c > t ? 0.0 : sh.p.x[t][c];
  }
  if (blk == 0 && wave == 0) {
    const double tol = (double)n * DBL_EPSILON * ajj;
    const unsigned long long bad = __ballot(col && (!(piv > tol) || !isfinite(piv)));
    const int fail = bad ? k0 + __ffsll((long long)bad) : 0;  // first failing column + 1
    if (lane == 0 && (s == 0 || fail)) a.info->fail_col = fail;
  }
}

// The tile at (r0, c0) of the lower triangle takes block column s - 1's update.
// The next launch's diagonal block goes to the rows 32 above its place, in the
// zero triangle: that launch's workgroups all read it, at any time while the
// first of them writes the factored block to L.  chol_clear zeroes it again.
__device__ void chol_update(const FactorArgs& a, int s, int r0, int c0, CholShared& sh) {
  const int n = a.n, kp = kBlk * (s - 1);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const double* __restrict__ src = s == 1 ? a.A : a.L;
  double* __restrict__ L = a.L;
  double la[64 * kBlk / 256], lb[64 * kBlk / 256];
#pragma unroll
  for (int u = 0; u < 64 * kBlk / 256; ++u) {
    const int i = 8 * u + threadIdx.x / kBlk, p = threadIdx.x % kBlk;
    la[u] = r0 + i < n ? L[(size_t)(r0 + i) * n + kp + p] : 0.0;
    lb[u] = c0 + i < n ? L[(size_t)(c0 + i) * n + kp + p] : 0.0;
  }
  // a wave's 16 rows: entry i of tile v: row 4 i + lane / 16, column 16 v + lane % 16
  const int i0 = r0 + 16 * wave + (lane >> 4), j0 = c0 + (lane & 15);
  f64x4 x[4];
#pragma unroll
  for (int v = 0; v < 4; ++v)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      x[v][i] = i0 + 4 * i < n && j0 + 16 * v <= i0 + 4 * i ? src[(size_t)(i0 + 4 * i) * n + j0 + 16 * v] : 0.0;
#pragma unroll
  for (int u = 0; u < 64 * kBlk / 256; ++u) {
    const int i = 8 * u + threadIdx.x / kBlk, p = threadIdx.x % kBlk;
    sh.u.a[i][p] = la[u];
    sh.u.b[i][p] = lb[u];
  }
  __syncthreads();
#pragma unroll
  for (int h = 0; h < kBlk; h += kPanel)
#pragma unroll
    for (int v = 0; v < 4; ++v) x[v] -= chain16(sh.u.a, 16 * wave, sh.u.b, 16 * v, h);
#pragma unroll
  for (int v = 0; v < 4; ++v)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = i0 + 4 * i, j = j0 + 16 * v;
      if (r < n && j <= r) {
        const int up = r < kBlk * (s + 2) ? kBlk : 0;
        L[(size_t)(r - up) * n + j] = x[v][i];
      }
    }
}

// v = L^T w (loading_of's sums) in pieces: piece k of block column b, its rows
// kLoadRows k .. from the diagonal block on, is launch b + 1 + k's, which adds it
// to what v holds of the pieces before.  Every piece up to the last block column's
// (factor_finish) has a launch, as a block column has one for each 32 of its
// rows.  The workgroup loads and multiplies, a lane per column adds up.  (One
// workgroup for a whole block column took longer than the panels: 11 us of a
// launch at n = 600, 17 at n = 1024.)
__host__ __device__ inline int chol_load_wgs(int n, int s) {
  // pieces k < s of block columns s - 1 - k with a row below n
  const int k = (n - kBlk * (s - 1) + kLoadRows - kBlk - 1) / (kLoadRows - kBlk);
  return s < k ? s : k;
}
__device__ void chol_loading(const FactorArgs& a, int b, int k, CholShared& sh) {
  const int n = a.n, c = threadIdx.x % kBlk, k0 = kBlk * b, i0 = k0 + kLoadRows * k;
  const double* __restrict__ col = a.L + k0 + c;
  constexpr int kPer = kLoadRows * kBlk / 256;
  double l[kPer], w[kPer];
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int i = i0 + 8 * u + threadIdx.x / kBlk;
    const bool on = i < n && i >= k0 + c;
    l[u] = on ? col[(size_t)i * n] : 0.0;
    w[u] = on ? a.w[i] : 0.0;
  }
#pragma unroll
  for (int u = 0; u < kPer; ++u) sh.prod[8 * u + threadIdx.x / kBlk][c] = l[u] * w[u];
  __syncthreads();
  if (threadIdx.x < kBlk) {
    // the entries above the diagonal and past row n are zeros here, and adding
    // one changes nothing
    double sum = k == 0 ? 0.0 : a.v64[k0 + c];
    for (int i = 0; i < kLoadRows; i += 32) {
      double p[32];
#pragma unroll
      for (int u = 0; u < 32; ++u) p[u] = sh.prod[i + u][c];
#pragma unroll
      for (int u = 0; u < 32; ++u) sum += p[u];
    }
    a.v64[k0 + c] = sum;
  }
}

// The place above the diagonal where block s waited (s >= 2).
__device__ void chol_clear(const FactorArgs& a, int s) {
  for (int e = threadIdx.x; e < kBlk * kBlk; e += blockDim.x) {
    const int j = kBlk * s + e % kBlk;
    if (j < a.n) a.L[(size_t)(kBlk * (s - 1) + e / kBlk) * a.n + j] = 0.0;
  }
}

// Launch 0 beside the first panel: the zero upper triangle of L, and the search
// of A's for non-finite entries (the factorisation itself meets those of the
// lower one).  One found poisons A's first entry, which the finishing kernel
// tests.
__device__ void chol_upper(const FactorArgs& a, int r0, int c0) {
  const int n = a.n;
  bool bad = false;
  for (int e = threadIdx.x; e < 64 * 64; e += blockDim.x) {
    const int i = r0 + e / 64, j = c0 + e % 64;
    if (i < n && j < n && j > i) {
      bad |= !isfinite(a.A[(size_t)i * n + j]);
      a.L[(size_t)i * n + j] = 0.0;
    }
  }
  if (bad) const_cast<double*>(a.A)[0] = __builtin_nan("");
}

__host__ __device__ inline int chol_panel_wgs(int n, int s) {
  const int below = n - kBlk * (s + 1);  // rows under the diagonal block
  return below > 0 ? (below + kBlk - 1) / kBlk : 1;
}
__host__ __device__ inline int chol_step_wgs(int n, int s) {
  if (kBlk * s >= n) return 0;
  const int t = s == 0 ? (n + 63) / 64 : (n - kBlk * (s + 1) + 63) / 64;
  return chol_panel_wgs(n, s) + (t > 0 ? (s == 0 ? t * t : t * (t + 1) / 2) : 0) + (s > 0 ? chol_load_wgs(n, s) : 0);
}

__device__ void chol_step(const FactorArgs& a, int s, CholShared& sh) {
  const int n = a.n, np = chol_panel_wgs(n, s);
  if ((int)blockIdx.x >= chol_step_wgs(n, s)) return;
  if (a.reuse) {
    // L is there from an earlier launch: the first panels' workgroups take a
    // block column's loading each, the last one left to factor_finish (where all
    // of them took 90 us of a serving round's setup at n = 600)
    const int b = blockIdx.x;
    if (s == 0 && kBlk * (b + 1) < n) {
      for (int k = 0; kBlk * b + kLoadRows * k < n; ++k) {
        if (k > 0) __syncthreads();
        chol_loading(a, b, k, sh);
      }
    }
    return;
  }
  if (s > 0) {
    // one read for the workgroup: the first one may be writing it
    if (threadIdx.x == 0) sh.failed = a.info->fail_col;
    __syncthreads();
    if (sh.failed != 0) return;  // a retry follows
  }
  if ((int)blockIdx.x < np) {
    chol_panel(a, s, blockIdx.x, sh);
    return;
  }
  if (s == 0) {
    const int t = blockIdx.x - np, nt = (n + 63) / 64;
    chol_upper(a, 64 * (t / nt), 64 * (t % nt));
    return;
  }
  const int nl = chol_load_wgs(n, s);
  if ((int)blockIdx.x < np + nl) {
    const int k = blockIdx.x - np;
    chol_loading(a, s - 1 - k, k, sh);
    if (k == 0 && s > 2) chol_clear(a, s - 1);
    return;
  }
  const int t = blockIdx.x - np - nl;
  int bi = (int)((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
  while (bi * (bi + 1) / 2 > t) --bi;
  while ((bi + 1) * (bi + 2) / 2 <= t) ++bi;
  const int bj = t - bi * (bi + 1) / 2, o = kBlk * (s + 1);
  chol_update(a, s, o + 64 * bi, o + 64 * bj, sh);
}

__global__ __launch_bounds__(256) void k_chol_step(FactorArgs a, int s) {
  __shared__ CholShared sh;
  chol_step(a, s, sh);
}
// blockIdx.y = query of a batch
__global__ __launch_bounds__(256) void k_chol_step_batch(const FactorArgs* fas, int s) {
  __shared__ CholShared sh;
  const FactorArgs a = fas[blockIdx.y];
  chol_step(a, s, sh);
}

template <int MAXN>
__device__ void factor_finish(const FactorArgs& a, FactorShared<MAXN>& sh) {
  const int tid = threadIdx.x;

  // Clear the query's accumulators.
  if (tid == 0) {
    DevAccum z = {};
    *a.acc = z;
  }
  for (int i = tid; i < kHistBins; i += blockDim.x) a.hist[i] = 0u;

  int attempts = 1, clamped = 0, last_fail = 0;
  double delta = 0.0;
  int j0 = kBlk * ((a.n - 1) / kBlk);  // the launches left this block column's loading
  if (a.reuse) {
    // L holds this covariance's factor from an earlier launch.
    const DevInfo fi = *a.finfo;
    attempts = fi.attempts;
    clamped = fi.clamped;
    last_fail = fi.fail_col;
    delta = fi.jitter;
    if (attempts < 0) {
      if (tid == 0) {
        a.info->attempts = -1;
        a.info->clamped = 0;
        a.info->fail_col = 0;
        a.info->jitter = 0.0;
      }
      return;
    }
  } else if (a.info->fail_col != 0 || !isfinite(a.A[0])) {
    __syncthreads();  // the record is read before anyone writes it
    if (!cholesky_body(a, sh, &attempts, &clamped, &last_fail, &delta)) return;
    j0 = 0;
  } else if (j0 > kBlk) {
    chol_clear(a, j0 / kBlk);
  }
  if (a.finfo && !a.reuse && tid == 0) {
    a.finfo->attempts = attempts;
    a.finfo->clamped = clamped;
    a.finfo->fail_col = last_fail;
    a.finfo->jitter = delta;
  }
  moments_body(a, sh.red, j0, attempts, clamped, last_fail, delta);
}

template <int MAXN>
__global__ __launch_bounds__(1024) void k_factor(FactorArgs a) {
  __shared__ FactorShared<MAXN> sh;
  factor_finish(a, sh);
}

// One workgroup per query of a batch (n <= MAXN).
template <int MAXN>
__global__ __launch_bounds__(1024) void k_factor_batch(const FactorArgs* fas) {
  __shared__ FactorShared<MAXN> sh;
  const FactorArgs a = fas[blockIdx.x];
  factor_finish(a, sh);
}

hipError_t launch_factor(const FactorArgs& a, hipStream_t stream) {
  if (a.n < 1 || a.n > kChunkMaxN) return hipErrorInvalidValue;
  for (int s = 0; kBlk * s < a.n; ++s)
    hipLaunchKernelGGL(k_chol_step, dim3(chol_step_wgs(a.n, s)), dim3(256), 0, stream, a, s);
  if (a.n <= kMaxN)
    hipLaunchKernelGGL(k_factor<kMaxN>, dim3(1), dim3(1024), 0, stream, a);
  else
    hipLaunchKernelGGL(k_factor<kChunkMaxN>, dim3(1), dim3(1024), 0, stream, a);
  return hipGetLastError();
}

// max_n: the batch's largest query (a panel of 78 KiB up to kMaxN, 99 KiB
// up to kBatchMaxN)
hipError_t launch_factor_batch(const FactorArgs* fas, int nq, int max_n, int fresh_n,
                               hipStream_t stream) {
  if (max_n < 1 || max_n > kBatchMaxN || fresh_n > max_n) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_chol_step_batch, dim3(chol_step_wgs(max_n, 0), nq), dim3(256), 0, stream, fas, 0);
  for (int s = 1; kBlk * s < fresh_n; ++s)
    hipLaunchKernelGGL(k_chol_step_batch, dim3(chol_step_wgs(fresh_n, s), nq), dim3(256), 0, stream, fas, s);
  if (max_n <= kMaxN)
    hipLaunchKernelGGL(k_factor_batch<kMaxN>, dim3(nq), dim3(1024), 0, stream, fas);
  else
    hipLaunchKernelGGL(k_factor_batch<kBatchMaxN>, dim3(nq), dim3(1024), 0, stream, fas);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Prep: layouts of the factor for the path kernels.
// ---------------------------------------------------------------------------
__device__ void prep_body(const PrepArgs& a, size_t gid, size_t gsz) {
  const int n = a.n;
  const double* __restrict__ L = a.L;
  if (a.s_hist) {
    for (size_t e = gid; e <= (size_t)n; e += gsz) a.s_hist[e] = 0ull;
  }
  if (a.v32) {
    for (size_t e = gid; e < (size_t)n; e += gsz) {
      a.v32[e] = (float)a.v64[e];
      a.mu32[e] = (float)a.mu[e];
    }
  }
  if (a.colpack) {
    // register kernel: column-packed lower triangle and loading
    for (size_t e = gid; e < (size_t)n; e += gsz)
      a.colpack[colpack_offset(n, (int)e) + n - (int)e] = (float)a.v64[e];
    for (size_t e = gid; e < (size_t)n * n; e += gsz) {
      const int i = (int)(e / n), j = (int)(e % n);
      if (j <= i) a.colpack[colpack_offset(n, j) + i - j] = (float)L[e];
    }
  }
  // MFMA: augmented rows (assets, zero pads, loss row 32T-1: -v and -w^T mu in
  // bf16 hi/lo parts; v and w^T mu in the fp32 wave kernel's, which negates the
  // sum as the register kernel does; likewise in the fp32 LDS kernel's unless
  // its tiles have no row to spare: row < n comes first)
  if (a.T > 0) {
    const int T = a.T, S = a.S;
    const float mp32 = (float)a.info->mp;
    auto entry = [&](int row, int k) {
      if (k >= n) return 0.0f;
      if (row < n) return k <= row ? (float)L[(size_t)row * n + k] : 0.0f;
      if (row == 32 * T - 1)
        return a.f32 ? (float)a.v64[k] : -(float)a.v64[k];
      return 0.0f;
    };
    for (size_t e = gid; e < (size_t)T * S * 64; e += gsz) {
      const int lane = (int)(e % 64);
      const int s = (int)((e / 64) % S);
      const int t = (int)(e / (64 * (size_t)S));
      const int row = 32 * t + (lane & 31);
      if (a.f32) {
        const int k0 = 8 * s + (lane >> 5);
        reinterpret_cast<float4*>(a.lfrag)[e] =
            make_float4(entry(row, k0), entry(row, k0 + 2), entry(row, k0 + 4), entry(row, k0 + 6));
        continue;
      }
      const int k0 = 16 * s + 8 * (lane >> 5);
      uint16_t hb[8], lb[8];
      for (int q = 0; q < 8; ++q) {
        const float m = entry(row, k0 + q);
        hb[q] = bf16_bits(m);
        lb[q] = bf16_bits(m - bf16_val(hb[q]));
      }
      uint4 h, l;
      h.x = hb[0] | ((uint32_t)hb[1] << 16);
      h.y = hb[2] | ((uint32_t)hb[3] << 16);
      h.z = hb[4] | ((uint32_t)hb[5] << 16);
      h.w = hb[6] | ((uint32_t)hb[7] << 16);
      l.x = lb[0] | ((uint32_t)lb[1] << 16);
      l.y = lb[2] | ((uint32_t)lb[3] << 16);
      l.z = lb[4] | ((uint32_t)lb[5] << 16);
      l.w = lb[6] | ((uint32_t)lb[7] << 16);
      a.lfrag[2 * e] = h;
      a.lfrag[2 * e + 1] = l;
    }
    for (size_t e = gid; e < (size_t)32 * T; e += gsz) {
      const int row = (int)e;
      a.rowinit[e] =
          row < n ? (float)a.mu[row]
                  : (row == 32 * T - 1 ? (a.f32 ? mp32 : -mp32) : INFINITY);
    }
  }
}

__global__ __launch_bounds__(256) void k_prep(PrepArgs a) {
  prep_body(a, (size_t)blockIdx.x * blockDim.x + threadIdx.x, (size_t)gridDim.x * blockDim.x);
}

// blockIdx.y = query of a batch
__global__ __launch_bounds__(256) void k_prep_batch(const PrepArgs* pas) {
  const PrepArgs a = pas[blockIdx.y];
  prep_body(a, (size_t)blockIdx.x * blockDim.x + threadIdx.x, (size_t)gridDim.x * blockDim.x);
}

hipError_t launch_prep_batch(const PrepArgs* pas, int nq, int max_n, hipStream_t stream) {
  int blocks = (max_n * max_n + 255) / 256;
  if (blocks > 256) blocks = 256;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(k_prep_batch, dim3(blocks, nq), dim3(256), 0, stream, pas);
  return hipGetLastError();
}

hipError_t launch_prep(const PrepArgs& a, hipStream_t stream) {
  const size_t work = (size_t)a.n * a.n;
  int blocks = (int)((work + 255) / 256);
  if (blocks > 1024) blocks = 1024;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(k_prep, dim3(blocks), dim3(256), 0, stream, a);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Collect: a query's record, S histogram and window losses to pinned host memory
// (block 0: the records; the others: kCollectBlocks per window).  One launch in
// place of a copy each, and the windows' lengths are read where they are.
// ---------------------------------------------------------------------------
constexpr int kCollectBlocks = 16;

__global__ __launch_bounds__(256) void k_collect(CollectArgs a) {
  const int tid = threadIdx.x;
  if (blockIdx.x == 0) {
    auto copy = [&](void* dst, const void* src, size_t bytes) {
      for (size_t i = tid; i < bytes / 4; i += 256)
        static_cast<uint32_t*>(dst)[i] = static_cast<const uint32_t*>(src)[i];
    };
    static_assert(sizeof(DevInfo) % 4 == 0 && sizeof(DevAccum) % 4 == 0, "copied as words");
    copy(a.h_info, a.info, sizeof(DevInfo));
    copy(a.h_acc, a.acc, sizeof(DevAccum));
    if (a.s_hist) copy(a.h_hist, a.s_hist, (size_t)(a.n + 1) * sizeof(unsigned long long));
    return;
  }
  const int al = (blockIdx.x - 1) / kCollectBlocks, part = (blockIdx.x - 1) % kCollectBlocks;
  const unsigned long long g = a.acc->gathered[al];
  const unsigned lim = a.cap < a.gather_cap ? a.cap : a.gather_cap;
  const unsigned cnt = g < lim ? (unsigned)g : lim;
  for (unsigned i = part * 256 + tid; i < cnt; i += kCollectBlocks * 256)
    a.h_win[(size_t)al * a.cap + i] = a.gather[(size_t)al * a.gather_cap + i];
}

hipError_t launch_collect(const CollectArgs& a, hipStream_t stream) {
  hipLaunchKernelGGL(k_collect, dim3(1 + kCollectBlocks * a.n_alpha), dim3(256), 0, stream, a);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Debug: the normal stream itself, one path per lane.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_normals(uint64_t seed, uint64_t path0, uint64_t npaths,
                                                 int n, float* out) {
  const uint64_t q = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= npaths) return;
  const Key2 key = key_of(seed);
  for (int b = 0; 4 * b < n; ++b) {
    float z[4];
    normals4(key, path0 + q, (uint32_t)b, z);
    for (int u = 0; u < 4; ++u)
      if (4 * b + u < n) out[q * n + 4 * b + u] = z[u];
  }
}

hipError_t launch_normals(uint64_t seed, uint64_t path0, uint64_t npaths, int n, float* out,
                          hipStream_t stream) {
  const uint64_t blocks = (npaths + 255) / 256;
  hipLaunchKernelGGL(k_normals, dim3((unsigned)blocks), dim3(256), 0, stream, seed, path0, npaths,
                     n, out);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Dispatch.
// ---------------------------------------------------------------------------
static uint64_t min_u64(uint64_t x, uint64_t y) { return x < y ? x : y; }

// Kept in an array, not on the heap: the allocation-free entry point asks too.  It
// holds every shape there is (about 70: a path kernel's block and LDS follow from
// n); past its end the runtime is asked again each time.
int resident_blocks(const void* kernel, int block, size_t lds) {
  struct Known {
    const void* kernel;
    int block;
    size_t lds;
    int per_cu;
  };
  static std::mutex mu;
  static Known known[128];
  static int count = 0;
  std::lock_guard<std::mutex> lk(mu);
  for (int i = 0; i < count; ++i)
    if (known[i].kernel == kernel && known[i].block == block && known[i].lds == lds) return known[i].per_cu;
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, block, lds) != hipSuccess ||
      per_cu < 1) {
    (void)hipGetLastError();
    per_cu = 1;
  }
  if (count < (int)(sizeof(known) / sizeof(known[0]))) known[count++] = {kernel, block, lds, per_cu};
  return per_cu;
}

// The path kernels' dynamic LDS past 64 KiB, which a device takes only as an
// attribute of the kernel: the largest request of each that has one.  Static LDS
// comes on top (160 KiB in all).
hipError_t init_path_kernels() {
  auto allow = [](PathKernel k, size_t lds) {
    return hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  };
  hipError_t e = allow(wave_kernel(kMfmaMaxT), wave_lds(kMfmaMaxT, 4 * kMfmaMaxT));
  for (int n : {kMaxN, 256, 128})  // 16, 8 and 4 waves
    if (e == hipSuccess) e = allow(f32_shape(n).kernel, f32_shape(kMaxN).lds);
  for (int T : {8, kStageMaxT})  // whole chunks and the histogram
    if (e == hipSuccess)
      e = allow(stage_shape(32 * T - 1, T, 2 * T).kernel, stage_cap(stage_waves(T)) * 4096 + (32 * T + 4) * 4);
  return e;
}

hipError_t launch_paths(int kernel, const PathArgs& a, int num_cus, hipStream_t stream) {
  if (a.npaths == 0) return hipSuccess;
  if (kernel == 3) {
    PathKernel k = mfma_kernel(a.n, a.T);
    if (!k) return hipErrorInvalidValue;
    const uint64_t blocks = min_u64((a.npaths + 255) / 256, (uint64_t)num_cus * 8);
    hipLaunchKernelGGL(k, dim3((unsigned)blocks), dim3(256), 0, stream, a);
    return hipGetLastError();
  }
  if (a.f32 == kF32Wave) {
    PathKernel k = wave_kernel(a.T);
    const size_t lds = wave_lds(a.T, a.S);
    const uint64_t per_cu = (uint64_t)resident_blocks((const void*)k, 256, lds);
    const uint64_t blocks = min_u64((a.npaths + 255) / 256, (uint64_t)num_cus * per_cu);
    hipLaunchKernelGGL(k, dim3((unsigned)blocks), dim3(256), lds, stream, a);
    return hipGetLastError();
  }
  if (a.f32 == kF32Lds) {
    if (a.n < 1 || a.n > kChunkMaxN) return hipErrorInvalidValue;
    const F32Shape s = f32_shape(a.n);
    const uint64_t blocks = min_u64((a.npaths + 63) / 64, (uint64_t)num_cus * s.per_cu);
    hipLaunchKernelGGL(s.kernel, dim3((unsigned)blocks), dim3(64 * s.waves), s.lds, stream, a);
    return hipGetLastError();
  }
  if (kernel == 1) {
    PathKernel k = reg_kernel(a.n);
    if (!k) return hipErrorInvalidValue;
    const uint64_t blocks = min_u64((a.npaths + 255) / 256, (uint64_t)num_cus * 8);
    hipLaunchKernelGGL(k, dim3((unsigned)blocks), dim3(256), 0, stream, a);
    return hipGetLastError();
  }
  if (kernel == 4) {
    if (a.n > kMfmaLdsMaxN) return hipErrorInvalidValue;
    if (a.T > 4 && a.T <= kStageMaxT) {
      const StageShape s = stage_shape(a.n, a.T, a.S);
      const uint64_t blocks = min_u64((a.npaths + 63) / 64, (uint64_t)num_cus * s.per_cu);
      hipLaunchKernelGGL(s.kernel, dim3((unsigned)blocks), dim3(64 * s.waves), s.lds, stream, a);
      return hipGetLastError();
    }
    PathKernel k = mfma_big_kernel(a.T);
    if (!k) return hipErrorInvalidValue;
    const int block = 64 * big_waves(a.T);
    const uint64_t per_cu = (uint64_t)resident_blocks((const void*)k, block);
    const uint64_t blocks = min_u64((a.npaths + 63) / 64, (uint64_t)num_cus * per_cu);
    hipLaunchKernelGGL(k, dim3((unsigned)blocks), dim3(block), 0, stream, a);
    return hipGetLastError();
  }
  return hipErrorInvalidValue;
}

}  // namespace mcr
