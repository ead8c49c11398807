// mcr_wave.hip -- the fp32 MFMA path kernel for n <= 127 (no barriers).
#include "mcr_kern_common.h"

namespace mcr {

// ---------------------------------------------------------------------------
// A wave runs 64 paths, one per lane, against T tiles of 32 rows (assets, +inf
// pads, loss row 32T-1) as two 32-path column tiles A (lanes 0-31's paths) and
// B (lanes 32-63's).  Every lane generates its own path's normals, so a step's
// Philox blocks are uniform over the wave (their share of the first two rounds
// runs on the scalar unit) and no lane idles at a ragged block count; one
// v_permlane32_swap per operand register pair then turns "the lane's normals"
// into the operands of both column tiles, and each factor fragment serves
// both.
// v_mfma_f32_32x32x2_f32 accumulates k = 0, 1 as two fused multiply-adds in that
// order, so a row's sum is the fmaf chain over ascending columns that the
// register kernel and the C mirror compute, bit for bit, without the scalar
// loads of the factor and their half-rate issue.
// Tile t only meets columns below 32 (t + 1) (the last tile, with the loss
// row, all of them): phase p handles columns 32p .. 32p + 31 for tiles p .. T-1.
// The workgroup's waves read the factor fragments and the rows' initial values
// from LDS, where they are staged once per query: from L2 the loads of a step
// cost more than its products (waves that started together wait together).
// D[row][path]: lane l holds rows 8(r/4) + 4(l/32) + r%4 of its column; two
// more swaps bring the counts and the loss back to the path's lane.
// Bound: the fp32 matrix instructions (64 cycles for 2 x 32 x 32 multiply-adds)
// and the vector instructions do not overlap on a SIMD (counted: no cycle with
// both, at n = 100 55 % with the former and 40 % with the latter), so a group costs
// both in full: at n = 127 320 of the former and 32
// blocks of normals; 4.62 ms for 1.9e7 paths, 8.76 ms in the tile kernel.
// ---------------------------------------------------------------------------
template <int T>
struct WaveAcc {
  f32x16 a[T], b[T];
};

template <int T>
__device__ __forceinline__ void init_rows(WaveAcc<T>& acc, const float4* rinit, int h) {
#pragma unroll
  for (int t = 0; t < T; ++t) {
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      const float4 v = rinit[8 * t + 2 * r4 + h];
      acc.a[t][4 * r4 + 0] = v.x;
      acc.a[t][4 * r4 + 1] = v.y;
      acc.a[t][4 * r4 + 2] = v.z;
      acc.a[t][4 * r4 + 3] = v.w;
    }
    acc.b[t] = acc.a[t];
  }
}

// Philox blocks 2o, 2o + 1 (8 columns, four 2-wide steps) through tiles
// P .. T-1; a FULL octet has all 8.  Fragments: [tile][octet][lane] float4,
// element e = L[row 32t + lane % 32][column 8o + 2e + lane / 32].
template <int T, int P, bool FULL>
__device__ __forceinline__ void octet_f32(WaveAcc<T>& acc, const PathArgs& a,
                                          const float4* frag, int o, Key2 key,
                                          PhiloxPath pp, uint32_t path_hi) {
  float4 f[T];
#pragma unroll
  for (int t = P; t < T; ++t) f[t] = frag[(t * a.S + o) * 64];
  float z[2][4];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int b = 2 * o + u;
    if (FULL || 4 * b + 2 < a.n) {
      normals4(key, pp, philox_block((uint32_t)b, path_hi, key), z[u]);
    } else if (4 * b < a.n) {
      normals2(key, pp, philox_block((uint32_t)b, path_hi, key), z[u]);
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (!FULL && 8 * o + 2 * e >= a.n) break;
    float &za = z[e >> 1][2 * (e & 1)], &zb = z[e >> 1][2 * (e & 1) + 1];
    swap32(za, zb);
#pragma unroll
    for (int t = P; t < T; ++t) {
      const float l = e == 0 ? f[t].x : e == 1 ? f[t].y : e == 2 ? f[t].z : f[t].w;
      acc.a[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(l, za, acc.a[t], 0, 0, 0);
      acc.b[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(l, zb, acc.b[t], 0, 0, 0);
    }
  }
}

// Phases P .. T-1 (32 (T - 1) <= n < 32 T, so only the last phase is ragged).
template <int T, int P>
__device__ __forceinline__ void run_phases(WaveAcc<T>& acc, const PathArgs& a, const float4* lds,
                                           int lane, Key2 key, PhiloxPath pp, uint32_t path_hi) {
  if constexpr (P < T) {
    const float4* frag = lds + lane;
    const int o1 = P == T - 1 ? a.n / 8 : 4 * P + 4;
#pragma unroll 1
    for (int o = 4 * P; o < o1; ++o) octet_f32<T, P, true>(acc, a, frag, o, key, pp, path_hi);
    if (P == T - 1 && (a.n & 7)) octet_f32<T, P, false>(acc, a, frag, o1, key, pp, path_hi);
    run_phases<T, P + 1>(acc, a, lds, lane, key, pp, path_hi);
  }
}

// The workgroup's copy of the factor fragments and row initial values.
template <int T>
__device__ __forceinline__ void stage_query(const PathArgs& a, float4* lds) {
  const int words = T * a.S * 64;
  for (int i = threadIdx.x; i < words; i += blockDim.x)
    lds[i] = reinterpret_cast<const float4*>(a.lfrag)[i];
  for (int i = threadIdx.x; i < 8 * T; i += blockDim.x)
    lds[words + i] = reinterpret_cast<const float4*>(a.rowinit)[i];
}

// Groups g0, g0 + gstep, ... < g1 of 64 paths of query a (staged at lds),
// accumulated into the tally t (no workgroup barriers).
template <int T>
__device__ __forceinline__ void wave_groups(const PathArgs& a, const float4* lds, uint64_t g0,
                                            uint64_t g1, uint64_t gstep, LdsTally<kTallySlots>* t, unsigned* sh_hist) {
  const int lane = threadIdx.x & 63, h = lane >> 5;
  const Key2 key = key_of(a.seed);
  const bool want_near = a.thr_lo < a.thr_hi;
  for (uint64_t grp = g0; grp < g1; grp += gstep) {
    const uint64_t first = a.path0 + grp * 64, path = first + lane, q = grp * 64 + lane;
    const PhiloxPath pp = philox_path((uint32_t)path, key);
    // the paths' high word is uniform except in a group that crosses a
    // multiple of 2^32, which runs once per high word for the lanes it fits
    uint32_t hi = (uint32_t)(first >> 32);
    for (;;) {
      const uint32_t path_hi = __builtin_amdgcn_readfirstlane(hi);
      WaveAcc<T> acc;
      init_rows<T>(acc, lds + T * a.S * 64, h);
      run_phases<T, 0>(acc, a, lds, lane, key, pp, path_hi);
      uint32_t ca = 0, cb = 0, na = 0, nb = 0;
#pragma unroll
      for (int tt = 0; tt < T; ++tt)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const bool excl = tt == T - 1 && r == 15 && h == 1;  // the loss row
          ca += (acc.a[tt][r] < a.thr && !excl) ? 1u : 0u;
          cb += (acc.b[tt][r] < a.thr && !excl) ? 1u : 0u;
        }
      if (want_near) {
#pragma unroll
        for (int tt = 0; tt < T; ++tt)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const bool excl = tt == T - 1 && r == 15 && h == 1;
            na |= acc.a[tt][r] >= a.thr_lo && acc.a[tt][r] <= a.thr_hi && !excl;
            nb |= acc.b[tt][r] >= a.thr_lo && acc.b[tt][r] <= a.thr_hi && !excl;
          }
        swap32(na, nb);
      }
      swap32(ca, cb);
      float la = acc.a[T - 1][15], lb = acc.b[T - 1][15];  // row 32T - 1 in the upper half-wave
      swap32(la, lb);
      tally_wave(a, t, q, (uint32_t)(path >> 32) == path_hi && q < a.npaths, (int)(ca + cb),
                 -lb, (na | nb) != 0, sh_hist);
      if (path_hi == (uint32_t)((first + 63) >> 32)) break;
      hi = path_hi + 1;
    }
  }
}

// waves per SIMD the registers must leave room for (issue pairs two waves, so
// four or two)
constexpr int wave_min_waves(int T) { return T <= 2 ? 4 : 2; }

template <int T>
__global__ __launch_bounds__(256, wave_min_waves(T)) void k_wave(PathArgs a) {
  extern __shared__ float4 lds[];
  __shared__ unsigned sh_hist[32 * kMfmaMaxT];
  __shared__ LdsTally<kTallySlots> t;
  const int n = a.n;
  const bool want_hist = a.s_hist != nullptr;
  if (want_hist) {
    for (int i = threadIdx.x; i <= n; i += blockDim.x) sh_hist[i] = 0u;
  }
  clear_tally(&t);
  stage_query<T>(a, lds);
  __syncthreads();
  const uint64_t waves = (uint64_t)gridDim.x * (blockDim.x >> 6);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  wave_groups<T>(a, lds, (uint64_t)blockIdx.x * (blockDim.x >> 6) + wave, (a.npaths + 63) / 64,
                      waves, &t, want_hist ? sh_hist : nullptr);
  __syncthreads();
  flush_tally_lds(a, &t, threadIdx.x);
  if (want_hist) {
    for (int i = threadIdx.x; i <= n; i += blockDim.x)
      if (sh_hist[i]) atomicAdd(&a.s_hist[i], (unsigned long long)sh_hist[i]);
  }
}

size_t wave_lds(int T, int S) { return sizeof(float4) * (size_t)(T * S * 64 + 8 * T); }

PathKernel wave_kernel(int T) {
  static const PathKernel k[kMfmaMaxT] = {k_wave<1>, k_wave<2>, k_wave<3>, k_wave<4>};
  return T >= 1 && T <= kMfmaMaxT ? k[T - 1] : nullptr;
}

}  // namespace mcr
