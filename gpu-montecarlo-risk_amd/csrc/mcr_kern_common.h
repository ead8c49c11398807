// mcr_kern_common.h -- device helpers shared by the path kernels: scalar
// views of read-only inputs, wave reductions, per-path tallies (crash count,
// VaR window bookkeeping, refinement histogram) and their flush.
#pragma once
#include <float.h>
#include <math.h>

#include <algorithm>

#include "mcr_internal.h"
#include "mcr_rng.h"

namespace mcr {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
#define MCR_CONSTP(T) const __attribute__((address_space(4))) T*

// Read-only inputs viewed through the constant address space: uniform reads
// become scalar loads whose results feed VALU ops as SGPR operands.
template <typename T>
__device__ __forceinline__ MCR_CONSTP(T) cview(const T* p) {
  return (MCR_CONSTP(T))p;
}

// A read-only struct loaded word by word through the constant address space
// (scalar loads when the address is uniform).
template <typename T>
__device__ __forceinline__ T load_const(const T* p) {
  static_assert(sizeof(T) % 4 == 0, "word-sized struct expected");
  uint32_t w[sizeof(T) / 4];
  MCR_CONSTP(uint32_t) src = cview(reinterpret_cast<const uint32_t*>(p));
#pragma unroll
  for (int i = 0; i < (int)(sizeof(T) / 4); ++i) w[i] = src[i];
  return __builtin_bit_cast(T, w);
}

__device__ __forceinline__ uint32_t wave_sum_u32(uint32_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}
__device__ __forceinline__ long long wave_sum_i64(long long v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}
__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// Loss -> fixed point in units of 2^-32, truncating (exact for |loss| >= 2^-9).
__device__ __forceinline__ long long fixed32(float v) {
  return (long long)((double)v * 4294967296.0);
}

struct LaneTally {
  uint32_t count;
  uint32_t near;
  uint32_t above[kMaxAlpha];
  long long sum_above[kMaxAlpha];
  uint32_t hist_below, hist_above;
};

// Wave-aggregated append of losses that fall inside window `al`.
__device__ __forceinline__ void append_loss(const PathArgs& a, int al, bool in, float v) {
  const unsigned long long m = __ballot(in);
  if (m == 0ull) return;
  const int lane = __lane_id();
  const int leader = __ffsll((long long)m) - 1;
  // set bits of m below this lane, counted by mbcnt: the mask by a 64-bit shift
  // gave wrong ranks where the compiler had put the lane index, its shift
  // amount, into the last register of the wave's allocation (two losses of a
  // wave then shared a slot)
  const unsigned rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                  __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
  unsigned long long base = 0;
  if (lane == leader) base = atomicAdd(&a.acc->gathered[al], (unsigned long long)__popcll(m));
  base = __shfl(base, leader);
  if (in) {
    const unsigned long long idx = base + rank;
    if (idx < a.gather_cap) a.gather[(size_t)al * a.gather_cap + idx] = v;
  }
}

// Per-path bookkeeping shared by every path kernel.  Lanes that reach it are
// active paths; ballots inside see exactly those lanes.
// Window bounds are re-read from the (scalar-cached) info block each path
// rather than held in SGPRs across the path loop.
__device__ __forceinline__ void tally_path(const PathArgs& a, LaneTally& t, uint64_t q, int S,
                                           float loss, bool near, unsigned* sh_hist) {
  const DevInfo* ip = a.info;
  asm volatile("" : "+s"(ip));
  MCR_CONSTP(DevInfo) w = cview(ip);
  t.count += (S >= a.k) ? 1u : 0u;
  t.near += near ? 1u : 0u;
  if (a.S_out) a.S_out[q] = S;
  if (a.loss_out) a.loss_out[q] = loss;
  if (sh_hist) atomicAdd(&sh_hist[S], 1u);
  if (a.loss_mode == kLossBracket) {
#pragma unroll
    for (int al = 0; al < kMaxAlpha; ++al) {
      if (al < a.n_alpha) {
        if (loss > w->hi[al]) {
          t.above[al] += 1u;
          t.sum_above[al] += fixed32(loss);
        }
        append_loss(a, al, loss >= w->lo[al] && loss <= w->hi[al], loss);
      }
    }
  } else if (a.loss_mode == kLossHist) {
    const float pos = (loss - w->hist_lo) * w->hist_scale;
    if (!(pos >= 0.0f)) {  // also catches NaN
      t.hist_below += 1u;
    } else if (!(pos < (float)kHistBins)) {
      t.hist_above += 1u;
    } else {
      atomicAdd(&a.hist[(int)pos], 1u);
    }
  }
}

__device__ __forceinline__ void flush_tally(const PathArgs& a, const LaneTally& t) {
  const int lane = __lane_id();
  const uint32_t c = wave_sum_u32(t.count);
  const uint32_t nr = wave_sum_u32(t.near);
  if (lane == 0) {
    if (c) atomicAdd(&a.acc->count, (unsigned long long)c);
    if (nr) atomicAdd(&a.acc->near, (unsigned long long)nr);
  }
  if (a.loss_mode == kLossBracket) {
#pragma unroll
    for (int al = 0; al < kMaxAlpha; ++al) {
      if (al < a.n_alpha) {
        const uint32_t ab = wave_sum_u32(t.above[al]);
        const long long sm = wave_sum_i64(t.sum_above[al]);
        if (lane == 0 && ab) {
          atomicAdd(&a.acc->above[al], (unsigned long long)ab);
          atomicAdd((unsigned long long*)&a.acc->sum_above[al], (unsigned long long)sm);
        }
      }
    }
  } else if (a.loss_mode == kLossHist) {
    const uint32_t b = wave_sum_u32(t.hist_below);
    const uint32_t ab = wave_sum_u32(t.hist_above);
    if (lane == 0) {
      if (b) atomicAdd(&a.acc->hist_below, (unsigned long long)b);
      if (ab) atomicAdd(&a.acc->hist_above, (unsigned long long)ab);
    }
  }
}

// The same tallies for kernels whose waves finish 64 paths at once: kept in LDS
// (ballots and population counts, added by one lane; the losses above a window
// add themselves), so a path loop carries none of them in registers.  One record
// per workgroup.  LDS takes adds to one address in turn, so kernels with the LDS
// to spare spread the lanes' losses over SLOTS sums: at a level of 5 % 60 of the
// 64 lanes add one.
template <int SLOTS>
struct LdsTally {
  unsigned long long v[4 + kMaxAlpha];  // count, near, hist below / above, above[]
  unsigned long long sum_above[kMaxAlpha][SLOTS];
};

// SLOTS of the kernels for n <= 127, whose LDS is free (1e7-2e7 paths, level 5 %, 1
// -> 16 slots: n = 8 665 -> 439 us, n = 20 805 -> 582, n = 50 715 -> 600; at 99 %
// the same; 32 no better).  The ones past n = 127 fill it, and have a tenth of the
// losses for their work: one.
constexpr int kTallySlots = 16;

// By a thread per word.
template <int SLOTS>
__device__ __forceinline__ void clear_tally(LdsTally<SLOTS>* t) {
  constexpr int kWords = sizeof(LdsTally<SLOTS>) / 8;
  static_assert(kWords <= 256, "a word per thread");
  if (threadIdx.x < kWords) reinterpret_cast<unsigned long long*>(t)[threadIdx.x] = 0ull;
}

// All 64 lanes of the wave, valid marking the paths that count.
template <int SLOTS>
__device__ __forceinline__ void tally_wave(const PathArgs& a, LdsTally<SLOTS>* t, uint64_t q, bool valid,
                                           int S, float loss, bool near, unsigned* sh_hist) {
  const DevInfo* ip = a.info;
  asm volatile("" : "+s"(ip));
  MCR_CONSTP(DevInfo) w = cview(ip);
  auto add = [&](int slot, bool on) {
    const unsigned long long m = __ballot(on);
    if (m != 0ull && __lane_id() == 0) atomicAdd(&t->v[slot], (unsigned long long)__popcll(m));
  };
  add(0, valid && S >= a.k);
  if (a.thr_lo < a.thr_hi) add(1, valid && near);
  if (valid) {
    if (a.S_out) a.S_out[q] = S;
    if (a.loss_out) a.loss_out[q] = loss;
    if (sh_hist) atomicAdd(&sh_hist[S], 1u);
  }
  if (a.loss_mode == kLossBracket) {
#pragma unroll
    for (int al = 0; al < kMaxAlpha; ++al) {
      if (al < a.n_alpha) {
        const bool above = valid && loss > w->hi[al];
        add(4 + al, above);
        if (above)
          atomicAdd(&t->sum_above[al][threadIdx.x % SLOTS], (unsigned long long)fixed32(loss));
        append_loss(a, al, valid && loss >= w->lo[al] && loss <= w->hi[al], loss);
      }
    }
  } else if (a.loss_mode == kLossHist) {
    const float pos = (loss - w->hist_lo) * w->hist_scale;
    const bool below = !(pos >= 0.0f);  // also catches NaN
    const bool past = !below && !(pos < (float)kHistBins);
    add(2, valid && below);
    add(3, valid && past);
    if (valid && !below && !past) atomicAdd(&a.hist[(int)pos], 1u);
  }
}

// Lane i of the first 12 adds tally i to the query's accumulators and clears it.
template <int SLOTS>
__device__ __forceinline__ void flush_tally_lds(const PathArgs& a, LdsTally<SLOTS>* t, int i) {
  if (i >= 4 + 2 * kMaxAlpha) return;
  unsigned long long* const acc = &a.acc->count;
  // DevAccum: count, near, above[], sum_above[], gathered[], hist below, hist above
  unsigned long long* dst = i < 2 ? acc + i
                            : i < 4 ? &a.acc->hist_below + (i - 2)
                                    : acc + (i - 2);
  unsigned long long v = 0;
  if (i < 4 + kMaxAlpha) {
    v = t->v[i];
    t->v[i] = 0ull;
  } else {
    unsigned long long* sum = t->sum_above[i - 4 - kMaxAlpha];
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) v += sum[s];
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) sum[s] = 0ull;
  }
  if (v) atomicAdd(dst, v);
}

// Workgroup form of flush_tally for kernels whose waves all tally paths: each
// wave sums its lanes, the waves' sums meet in LDS, and wave 0 issues one
// atomic per counter for the whole workgroup (a per-wave flush costs every
// wave its own L2 atomics: at 8 waves per CU they were most of the launch's
// HBM write traffic).  Every thread of the workgroup must call it (barrier).
__device__ __forceinline__ void flush_tally_block(const PathArgs& a, const LaneTally& t) {
  constexpr int kWaves = 16;              // workgroups of up to 1024 threads
  constexpr int kU = 4 + kMaxAlpha;       // count, near, hist below/above, above[]
  __shared__ uint32_t s_u[kWaves][kU];
  __shared__ long long s_l[kWaves][kMaxAlpha];
  const int lane = __lane_id(), wave = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  const bool bracket = a.loss_mode == kLossBracket, hist = a.loss_mode == kLossHist;
  uint32_t u[kU];
  long long l[kMaxAlpha];
  u[0] = wave_sum_u32(t.count);
  u[1] = wave_sum_u32(t.near);
  u[2] = hist ? wave_sum_u32(t.hist_below) : 0u;
  u[3] = hist ? wave_sum_u32(t.hist_above) : 0u;
#pragma unroll
  for (int al = 0; al < kMaxAlpha; ++al) {
    const bool on = bracket && al < a.n_alpha;
    u[4 + al] = on ? wave_sum_u32(t.above[al]) : 0u;
    l[al] = on ? wave_sum_i64(t.sum_above[al]) : 0ll;
  }
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < kU; ++k) s_u[wave][k] = u[k];
#pragma unroll
    for (int al = 0; al < kMaxAlpha; ++al) s_l[wave][al] = l[al];
  }
  __syncthreads();
  if (wave == 0) {
    unsigned long long* const dst[kU] = {&a.acc->count, &a.acc->near, &a.acc->hist_below,
                                         &a.acc->hist_above, &a.acc->above[0], &a.acc->above[1],
                                         &a.acc->above[2], &a.acc->above[3]};
#pragma unroll
    for (int k = 0; k < kU; ++k) {
      const uint32_t v = wave_sum_u32(lane < nw ? s_u[lane][k] : 0u);
      if (lane == 0 && v) atomicAdd(dst[k], (unsigned long long)v);
    }
#pragma unroll
    for (int al = 0; al < kMaxAlpha; ++al) {
      if (bracket && al < a.n_alpha) {
        const long long v = wave_sum_i64(lane < nw ? s_l[lane][al] : 0ll);
        if (lane == 0 && v) atomicAdd((unsigned long long*)&a.acc->sum_above[al], (unsigned long long)v);
      }
    }
  }
}

__device__ __forceinline__ void zero_tally(LaneTally& t) {
  t.count = 0;
  t.near = 0;
#pragma unroll
  for (int i = 0; i < kMaxAlpha; ++i) {
    t.above[i] = 0;
    t.sum_above[i] = 0;
  }
  t.hist_below = 0;
  t.hist_above = 0;
}

__device__ __forceinline__ uint16_t bf16_bits(float f) {
  return __builtin_bit_cast(uint16_t, (__bf16)f);
}
__device__ __forceinline__ float bf16_val(uint16_t b) { return as_f32((uint32_t)b << 16); }


// Converted as a vector: one v_cvt_pk_bf16_f32 (two scalar conversions and
// their merge were four instructions).
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, bf16x2));
}

// z0, z1 -> their bf16 hi and lo parts, two per 32-bit word
__device__ __forceinline__ void split2(float z0, float z1, uint32_t* hi, uint32_t* lo) {
  const uint32_t h = pack_bf16x2(z0, z1);
  *hi = h;
  *lo = pack_bf16x2(z0 - as_f32(h << 16), z1 - as_f32(h & 0xffff0000u));
}

// z[0..7] -> bf16 hi and lo parts, two per 32-bit word
__device__ __forceinline__ void split8(const float* z, uint32_t hi[4], uint32_t lo[4]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) split2(z[2 * q], z[2 * q + 1], &hi[q], &lo[q]);
}

// lanes 32-63 of x <-> lanes 0-31 of y
__device__ __forceinline__ void swap32(uint32_t& x, uint32_t& y) {
  const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
  x = r[0];
  y = r[1];
}
__device__ __forceinline__ void swap32(float& x, float& y) {
  uint32_t u = as_u32(x), v = as_u32(y);
  swap32(u, v);
  x = as_f32(u);
  y = as_f32(v);
}

__device__ __forceinline__ bf16x8 as_bf16x8(const uint32_t w[4]) {
  return __builtin_bit_cast(bf16x8, make_uint4(w[0], w[1], w[2], w[3]));
}

// The row tiles of wave `wave` of NW (wave w runs on SIMD w % 4), at most SLOTS:
// tiles in descending order to the SIMD with the least work so far (tile t is
// t + 1 units) that has a slot free, there to its waves in turn.  tile[SLOTS - 1]
// is the wave's first (larger) one, -1 a free slot; tile T - 1 is wave 0's first.
template <int NW, int SLOTS>
__device__ __forceinline__ void deal_tiles(int T, int wave, int (&tile)[SLOTS]) {
  static_assert(SLOTS == 2, "a wave's two tiles");
  tile[0] = tile[1] = -1;
  int load[4] = {0, 0, 0, 0}, cnt[4] = {0, 0, 0, 0};
  for (int tt = T - 1; tt >= 0; --tt) {
    int s = -1, best = 1 << 30;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (cnt[k] < SLOTS * NW / 4 && load[k] < best) {
        s = k;
        best = load[k];
      }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (k == s) {
        // the waves take their second tiles in reverse order
        const int q = cnt[k], w = q < NW / 4 ? q : SLOTS * NW / 4 - 1 - q;
        if (k + 4 * w == wave) tile[q < NW / 4 ? 1 : 0] = tt;
        load[k] += tt + 1;
        cnt[k] = q + 1;
      }
    }
  }
  tile[0] = __builtin_amdgcn_readfirstlane(tile[0]);
  tile[1] = __builtin_amdgcn_readfirstlane(tile[1]);
}

typedef void (*PathKernel)(PathArgs);
PathKernel reg_kernel(int n);          // mcr_reg.hip
PathKernel wave_kernel(int T);         // mcr_wave.hip
PathKernel mfma_kernel(int n, int T);  // mcr_mfma.hip
// mcr_f32.hip: kernel, waves per workgroup, workgroups per CU, dynamic LDS
struct F32Shape {
  PathKernel kernel;
  int waves, per_cu;
  size_t lds;
};
F32Shape f32_shape(int n);
// mcr_stage.hip
// Steps that fit the LDS of one of the four (4 waves) or two (8) workgroups of a
// compute unit; a longer S is taken in equal chunks, the sums staying in registers.
__host__ __device__ constexpr int stage_cap(int waves) { return waves == 4 ? 9 : 19; }
constexpr int kStageMaxT = 16;  // row tiles
struct StageShape {
  PathKernel kernel;
  int waves, per_cu;
  size_t lds;
};
StageShape stage_shape(int n, int T, int S);
int stage_waves(int T);
BatchKernel batch_stage_kernel(int T);
PathKernel mfma_big_kernel(int T);     // mcr_mfma_big.hip

}  // namespace mcr
