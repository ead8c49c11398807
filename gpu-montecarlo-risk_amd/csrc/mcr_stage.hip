// mcr_stage.hip -- bf16x3 MFMA path kernel whose workgroup stages all normals of
// its 64 paths before it multiplies.
#include "mcr_kern_common.h"

namespace mcr {

// ---------------------------------------------------------------------------
// The operands, rows and sums of mcr_mfma_big.hip's kernels (same fragments, the
// same sequence of products into every accumulator, so the same bits), with two
// barriers per 64 paths instead of one per K step or two: the waves deal the
// Philox blocks and write the normals' bf16 parts to LDS as B operands of all S
// steps (4 KiB a step), and behind a barrier every wave runs its one or two row
// tiles through, fragments streamed from L2 two steps ahead.  Two or four
// workgroups per CU, so that one's normals run beside another's products.  Bound:
// the two units' work, which overlaps little: of the SIMD cycles at n = 143 / 301 /
// 400 the vector unit issues in 76 / 65 / 63 %, the matrix unit is busy in 22 / 34 /
// 40, both at once in 12 / 10 / 14, neither in 14 / 11 / 10.  Queries of 4e11 / (n^2 + 40 n) paths, against waves that generate and
// multiply in turn (n < 384) or take a role each: n = 143 3.16 -> 2.88 ms, n = 200
// 2.58 -> 2.46, n = 301 2.18 -> 1.99, n = 400 2.18 -> 1.81, n = 511 1.96 -> 1.71.
// Past 16 row tiles a CU holds one such workgroup, nothing runs beside it, and
// the split roles stay (n = 600 1.81 / 1.80).
// ---------------------------------------------------------------------------
constexpr int kStageSlots = 2;  // row tiles per wave: 64 accumulator registers
__host__ __device__ constexpr int stage_chunk(int S, int waves) {
  const int chunks = (S + stage_cap(waves) - 1) / stage_cap(waves);
  return (S + chunks - 1) / chunks;
}

struct StageAcc {
  f32x16 a[kStageSlots], b[kStageSlots];  // paths 0-31, 32-63
};

struct StageFrag {
  uint4 hi[kStageSlots], lo[kStageSlots];
};

template <int I>
__device__ __forceinline__ void stage_mul(StageAcc& acc, const StageFrag& f, const uint4* zs) {
  const bf16x8 ah = __builtin_bit_cast(bf16x8, zs[0]), al = __builtin_bit_cast(bf16x8, zs[64]);
  const bf16x8 bh = __builtin_bit_cast(bf16x8, zs[128]), bl = __builtin_bit_cast(bf16x8, zs[192]);
#pragma unroll
  for (int i = I; i < kStageSlots; ++i) {
    const bf16x8 hi = __builtin_bit_cast(bf16x8, f.hi[i]), lo = __builtin_bit_cast(bf16x8, f.lo[i]);
    acc.a[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lo, ah, acc.a[i], 0, 0, 0);
    acc.b[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lo, bh, acc.b[i], 0, 0, 0);
    acc.a[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hi, al, acc.a[i], 0, 0, 0);
    acc.b[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hi, bl, acc.b[i], 0, 0, 0);
    acc.a[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hi, ah, acc.a[i], 0, 0, 0);
    acc.b[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hi, bh, acc.b[i], 0, 0, 0);
  }
}

// Steps s0 .. s1 - 1 through the slots I .. kStageSlots-1; zs is the lane's place
// of step s0.  Two sets of fragment registers, each loaded again as soon as its
// step is multiplied.
template <int I>
__device__ __forceinline__ void stage_run(StageAcc& acc, const int (&tile)[kStageSlots], int S, int s0,
                                          int s1, const uint4* zs, __amdgpu_buffer_rsrc_t rs, int voff) {
  if (s0 >= s1) return;
  StageFrag f[2];
  auto load = [&](StageFrag& r, int s) {
#pragma unroll
    for (int i = I; i < kStageSlots; ++i) {
      const int o = (tile[i] * S + min(s, s1 - 1)) * 2048;
      r.hi[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rs, voff, o, 0));
      r.lo[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rs, voff + 16, o, 0));
    }
  };
  load(f[0], s0);
  load(f[1], s0 + 1);
  int s = s0;
#pragma unroll 1
  for (; s + 2 <= s1; s += 2) {
    stage_mul<I>(acc, f[0], zs + (s - s0) * 256);
    load(f[0], s + 2);
    stage_mul<I>(acc, f[1], zs + (s + 1 - s0) * 256);
    load(f[1], s + 3);
  }
  if (s < s1) stage_mul<I>(acc, f[0], zs + (s - s0) * 256);
}

template <int NW>
struct StageShared {
  int sS[NW][64];
  float sLoss[64];
  LdsTally<1> t;
};

// Groups g0, g0 + gstep, ... < g1 of 64 paths of query a; zs: [step][path half]
// [hi, lo][operand lane], S 256 entries.
template <int NW>
__device__ __forceinline__ void stage_groups(const PathArgs& a, uint64_t g0, uint64_t g1,
                                             uint64_t gstep, uint4* zs, StageShared<NW>& sh,
                                             unsigned* sh_hist) {
  const int lane = threadIdx.x & 63, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = a.n, T = a.T, S = a.S, nb = (n + 3) >> 2, chunk = stage_chunk(S, NW);
  int tile[kStageSlots];
  deal_tiles<NW, kStageSlots>(T, wave, tile);
  const int end0 = tile[0] < 0 ? 0 : min(2 * tile[0] + 2, S);
  const int end1 = tile[1] < 0 ? 0 : (tile[1] == T - 1 ? S : min(2 * tile[1] + 2, S));
  const Key2 key = key_of(a.seed);
  const float4* __restrict__ rinit = (const float4*)a.rowinit;
  const uint64_t fp = (uint64_t)a.lfrag;
  // through readfirstlane: uniform also where the record comes from memory
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(((uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(fp >> 32)) << 32) |
              (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)fp)),
      (short)0, __builtin_amdgcn_readfirstlane(T * S * 2048), 0x00020000);

  for (uint64_t grp = g0; grp < g1; grp += gstep) {
    const uint64_t first = a.path0 + grp * 64, path = first + lane, q = grp * 64 + lane;
    const PhiloxPath pp = philox_path((uint32_t)path, key);
    const uint32_t path_hi = __builtin_amdgcn_readfirstlane((uint32_t)(first >> 32));
    // all groups but one that crosses a multiple of 2^32
    const bool one_hi = __builtin_amdgcn_readfirstlane((uint32_t)first) <= 0xffffffffu - 63u;
    StageAcc acc;
    for (int sc = 0; sc < S; sc += chunk) {
      const int se = min(sc + chunk, S);
      for (int b = 4 * sc + wave; b < 4 * se; b += NW) {
        float z[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (b < nb) {
          if (one_hi)
            normals4(key, pp, philox_block((uint32_t)b, path_hi, key), z);
          else
            normals4(key, path, (uint32_t)b, z);
        }
        uint2 hi, lo;
        split2(z[0], z[1], &hi.x, &lo.x);
        split2(z[2], z[3], &hi.y, &lo.y);
        // normals 16 s + 4 u ..: operand lane path % 32 + 32 (u / 2), half u % 2
        const int u = b & 3;
        uint2* d = reinterpret_cast<uint2*>(zs + ((b >> 2) - sc) * 256 + h * 128 + (lane & 31) + 32 * (u >> 1)) + (u & 1);
        d[0] = hi;
        d[128] = lo;  // 64 operand lanes on
      }
      if (sc == 0) {
#pragma unroll
        for (int i = 0; i < kStageSlots; ++i) {
          if (tile[i] < 0) continue;
#pragma unroll
          for (int r4 = 0; r4 < 4; ++r4) {
            const float4 w = rinit[8 * tile[i] + 2 * r4 + h];
            acc.a[i][4 * r4 + 0] = w.x;
            acc.a[i][4 * r4 + 1] = w.y;
            acc.a[i][4 * r4 + 2] = w.z;
            acc.a[i][4 * r4 + 3] = w.w;
          }
          acc.b[i] = acc.a[i];
        }
      }
      __syncthreads();
      // products before another workgroup's normals: they fill the matrix unit
      // from few issue slots (1e12 / (n^2 + 40 n) paths: n = 143, 200 and 255 the
      // same, n = 301 4.85 -> 4.89 ms, n = 400 4.35 -> 4.23, n = 511 3.79 -> 3.71)
      __builtin_amdgcn_s_setprio(2);
      stage_run<0>(acc, tile, S, sc, min(end0, se), zs + lane, rs, 32 * lane);
      const int s1 = max(sc, end0);
      stage_run<1>(acc, tile, S, s1, min(end1, se), zs + (s1 - sc) * 256 + lane, rs, 32 * lane);
      __builtin_amdgcn_s_setprio(0);
      if (se < S) __syncthreads();  // the chunk's normals are read
    }
    if (wave == 0) {
      float la = acc.a[1][15], lb = acc.b[1][15];
      swap32(la, lb);  // lb: row 32T - 1 of the lane's path
      sh.sLoss[lane] = lb;
    }
    uint32_t ca = 0, cb = 0;
#pragma unroll
    for (int i = 0; i < kStageSlots; ++i) {
      if (tile[i] < 0) continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const bool excl = r == 15 && h == 1 && i == 1 && wave == 0;  // the loss row
        ca += acc.a[i][r] < a.thr && !excl ? 1u : 0u;
        cb += acc.b[i][r] < a.thr && !excl ? 1u : 0u;
      }
    }
    swap32(ca, cb);
    sh.sS[wave][lane] = (int)(ca + cb);
    __syncthreads();
    if (wave == 0) {
      int tot = 0;
#pragma unroll
      for (int w = 0; w < NW; ++w) tot += sh.sS[w][lane];
      tally_wave(a, &sh.t, q, q < a.npaths, tot, sh.sLoss[lane], false, sh_hist);
    }
    // sS and sLoss are next written behind the next group's first barrier
  }
}

template <int NW>
__global__ __launch_bounds__(64 * NW, 4) void k_mfma_stage(PathArgs a) {
  extern __shared__ uint4 stage_z[];
  __shared__ StageShared<NW> sh;
  unsigned* sh_hist = reinterpret_cast<unsigned*>(stage_z + stage_chunk(a.S, NW) * 256);  // [n + 1]
  const bool want_hist = a.s_hist != nullptr;
  if (want_hist) {
    for (int i = threadIdx.x; i <= a.n; i += blockDim.x) sh_hist[i] = 0u;
  }
  clear_tally(&sh.t);
  __syncthreads();
  stage_groups<NW>(a, blockIdx.x, (a.npaths + 63) / 64, gridDim.x, stage_z, sh,
                   want_hist ? sh_hist : nullptr);
  __syncthreads();
  flush_tally_lds(a, &sh.t, threadIdx.x);
  if (want_hist) {
    for (int i = threadIdx.x; i <= a.n; i += blockDim.x)
      if (sh_hist[i]) atomicAdd(&a.s_hist[i], (unsigned long long)sh_hist[i]);
  }
}

// Persistent batch form (see mcr_mfma_big.hip's k_batch_paths): the workgroup
// takes items until the class's list is exhausted, its tally flushed after each.
template <int NW>
__global__ __launch_bounds__(64 * NW, 4) void k_batch_stage(BatchArgs b) {
  __shared__ uint4 zs[stage_cap(NW) * 256];
  __shared__ StageShared<NW> sh;
  __shared__ unsigned s_item;
  clear_tally(&sh.t);
  for (;;) {
    if (threadIdx.x == 0) s_item = atomicAdd(b.next, 1u);
    __syncthreads();
    const unsigned it = __builtin_amdgcn_readfirstlane(s_item);
    __syncthreads();
    if (it >= b.nitems) break;
    const WorkItem w = load_const(b.items + it);
    const PathArgs a = load_const(b.qs + w.query);
    stage_groups<NW>(a, w.first_group, w.first_group + w.ngroups, 1, zs, sh, nullptr);
    __syncthreads();
    flush_tally_lds(a, &sh.t, threadIdx.x);
  }
}

// Four waves reach 8 row tiles, eight 16.  Where both do (n = 128-255, S > 9) four
// in two chunks are the faster: 4e11 / (n^2 + 40 n) paths n = 159 2.63 / 2.72 ms,
// n = 200 2.46 / 2.54, n = 255 2.10 / 2.14.
int stage_waves(int T) { return T <= 8 ? 4 : 8; }

StageShape stage_shape(int n, int T, int S) {
  StageShape s;
  s.waves = stage_waves(T);
  s.per_cu = 16 / s.waves;  // four waves per SIMD
  s.lds = (size_t)stage_chunk(S, s.waves) * 4096 + ((n + 1) * sizeof(unsigned) + 15) / 16 * 16;
  s.kernel = s.waves == 8 ? k_mfma_stage<8> : k_mfma_stage<4>;
  return s;
}

BatchKernel batch_stage_kernel(int T) { return T <= 8 ? k_batch_stage<4> : k_batch_stage<8>; }

}  // namespace mcr
