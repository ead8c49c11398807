// mcr_f32.hip -- the fp32 MFMA path kernel for n > 127 (and any n up to 1024).
#include "mcr_kern_common.h"

namespace mcr {

// ---------------------------------------------------------------------------
// A workgroup of NW waves takes 64 paths, one per lane of a wave while it
// generates: the waves deal the Philox blocks and write the normals to LDS as
// operands of v_mfma_f32_32x32x2_f32 (octets of 8 columns, [octet][path half]
// [operand lane] float4, element e = column 8o + 2e + lane / 32 of path
// lane % 32 of the half).  After a barrier every wave runs its one or two
// 32-row tiles over the octets they reach (tile t: columns below 32 (t + 1)),
// factor fragments (1 KiB per tile and octet, for eight matrix instructions)
// streamed from L2 one octet ahead.  The instruction's two products are fused
// multiply-adds in ascending order, so a row sees mu_i, then z_0 .. z_i, as in
// the register kernel, bit for bit.  The loss row is the last tile's last row;
// where n is a multiple of 32 it would cost a tile of its own and is one fmaf
// chain per lane instead, by one wave before the products start (beside them
// each of its multiply-adds waits for a matrix instruction of the SIMD to end:
// n = 600 4.59 ms per 1.04e6 paths with the chain beside, 3.81 without it).
// Past kMaxN columns the normals no longer fit the LDS and are taken in chunks
// of kChunkCols, the accumulators staying in registers.
//
// Bound: the matrix instructions (64 cycles for 2 x 32 x 32 multiply-adds);
// vector instructions do not overlap them on a SIMD (counted: no cycle with both;
// n = 143 53 % matrix and 37 % vector, n = 300 67 and 26, n = 600 76 and 19), so the
// normals' time adds, and with no overlap to gain there is nothing to interleave: one barrier per
// chunk.  Tiles go to the four SIMDs largest first, to the least loaded one.
// Per 1e6 paths, this kernel against the vector kernels it replaced (tile to n =
// 608, column chunks past it): n = 143 0.35 / 0.56 ms, n = 300 1.03 / 2.15, n =
// 600 3.5 / 6.5, n = 1024 10.3 / 23.7; n = 600 is 103 TFLOP/s of n (n + 1) per
// path, two thirds of the matrix rate with the normals' time and the padded
// halves of the diagonal tiles in it.
// ---------------------------------------------------------------------------
constexpr int kChunkCols = 512;
constexpr int kSlots = 2;  // row tiles per wave: 64 accumulator registers, so that
                           // four waves fit a SIMD

struct F32Acc {
  f32x16 a[kSlots], b[kSlots];  // paths 0-31, 32-63
};

// Factor fragments through a buffer resource: the per-octet part of the address
// is a scalar offset (see mcr_mfma_big.hip).
__device__ __forceinline__ float4 load_frag(__amdgpu_buffer_rsrc_t rs, int voff, int tile, int S,
                                            int o) {
  return __builtin_bit_cast(float4,
                            __builtin_amdgcn_raw_buffer_load_b128(rs, voff, (tile * S + o) * 1024, 0));
}

// One octet (operands at zs) through the slots I .. kSlots-1.
template <int I>
__device__ __forceinline__ void mul_octet(F32Acc& acc, const float4 (&f)[kSlots], const float4* zs) {
  const float4 za = zs[0], zb = zs[64];
  const float a4[4] = {za.x, za.y, za.z, za.w}, b4[4] = {zb.x, zb.y, zb.z, zb.w};
#pragma unroll
  for (int e = 0; e < 4; ++e) {
#pragma unroll
    for (int i = I; i < kSlots; ++i) {
      const float l = e == 0 ? f[i].x : e == 1 ? f[i].y : e == 2 ? f[i].z : f[i].w;
      acc.a[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(l, a4[e], acc.a[i], 0, 0, 0);
      acc.b[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(l, b4[e], acc.b[i], 0, 0, 0);
    }
  }
}

// Octets o0 .. o1 - 1 through the slots I .. kSlots-1; zs is octet o0's place.
// D sets of fragment registers, each loaded again as soon as its octet is
// multiplied: the loads run D - 1 octets (512 cycles of one tile, at least)
// ahead, and no register is copied (a copy waits for its load).
template <int I, int D>
__device__ __forceinline__ void run_octets(F32Acc& acc, const int (&tile)[kSlots], int S, int o0,
                                           int o1, const float4* zs, __amdgpu_buffer_rsrc_t rs,
                                           int lane) {
  if (o0 >= o1) return;
  float4 f[D][kSlots];
  auto load = [&](float4 (&r)[kSlots], int o) {
#pragma unroll
    for (int i = I; i < kSlots; ++i) r[i] = load_frag(rs, 16 * lane, tile[i], S, min(o, o1 - 1));
  };
#pragma unroll
  for (int d = 0; d < D; ++d) load(f[d], o0 + d);
  int o = o0;
#pragma unroll 1
  for (; o + D <= o1; o += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      mul_octet<I>(acc, f[d], zs + (o + d - o0) * 128);
      load(f[d], o + d + D);
    }
  }
#pragma unroll
  for (int d = 0; d < D - 1; ++d)
    if (o + d < o1) mul_octet<I>(acc, f[d], zs + (o + d - o0) * 128);
}

template <int NW>
__global__ __launch_bounds__(64 * NW, 4) void k_f32_lds(PathArgs a) {
  extern __shared__ float4 zs[];  // [octet - chunk start][path half][64]
  __shared__ int sS[NW][64];
  __shared__ float sLoss[64];
  __shared__ LdsTally<1> t;
  const int n = a.n, T = a.T, S = a.S;
  const int nb = (n + 3) >> 2;
  const int chunk = n <= kMaxN ? S : kChunkCols / 8;  // octets
  unsigned* sh_hist = reinterpret_cast<unsigned*>(zs + chunk * 128);  // [n + 1]
  const int lane = threadIdx.x & 63, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool want_hist = a.s_hist != nullptr, want_near = a.thr_lo < a.thr_hi;
  if (want_hist) {
    for (int i = threadIdx.x; i <= n; i += blockDim.x) sh_hist[i] = 0u;
  }
  clear_tally(&t);

  int tile[kSlots];  // slot 1: the wave's first (larger) tile, T - 1 wave 0's
  deal_tiles<NW, kSlots>(T, wave, tile);
  // octets each slot runs: none, or its columns (0 <= end0 <= end1)
  const int end0 = tile[0] < 0 ? 0 : min(4 * tile[0] + 4, S);
  const int end1 = tile[1] < 0 ? 0 : min(4 * tile[1] + 4, S);
  const bool loss_row = (n & 31) != 0;

  const Key2 key = key_of(a.seed);
  const float mp32 = (float)cview(a.info)->mp;
  MCR_CONSTP(float) v = cview(a.v32);
  const float4* __restrict__ rinit = (const float4*)a.rowinit;
  const uint64_t fp = (uint64_t)a.lfrag;
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)fp, (short)0, T * S * 1024, 0x00020000);
  __syncthreads();

  for (uint64_t grp = blockIdx.x; grp * 64 < a.npaths; grp += gridDim.x) {
    const uint64_t first = a.path0 + grp * 64, path = first + lane, q = grp * 64 + lane;
    const PhiloxPath pp = philox_path((uint32_t)path, key);
    // the paths' high word is uniform except in a group that crosses a
    // multiple of 2^32, which runs once per high word for the lanes it fits
    uint32_t hi = (uint32_t)(first >> 32);
    for (;;) {
      const uint32_t path_hi = __builtin_amdgcn_readfirstlane(hi);
      F32Acc acc;
      float g = mp32;  // loss row: g = w^T mu + sum_j v_j z_j, j ascending
      for (int oc = 0; oc < S; oc += chunk) {
        const int oe = min(oc + chunk, S);
        for (int b = 2 * oc + wave; b < 2 * oe; b += NW) {
          float z[4] = {0.0f, 0.0f, 0.0f, 0.0f};
          if (b < nb) normals4(key, pp, philox_block((uint32_t)b, path_hi, key), z);
          // path p of half p / 32: even columns to operand lane p % 32, odd to 32 + p % 32
          float2* d = reinterpret_cast<float2*>(&zs[((b >> 1) - oc) * 128 + 64 * h + (lane & 31)]) + (b & 1);
          d[0] = make_float2(z[0], z[2]);
          d[64] = make_float2(z[1], z[3]);
        }
        if (oc == 0) {
#pragma unroll
          for (int i = 0; i < kSlots; ++i) {
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
        if (!loss_row) {
          if (wave == 0) {
#pragma unroll 4
            for (int o = oc; o < oe; ++o) {
              const float4* zp = &zs[(o - oc) * 128 + 64 * h + (lane & 31)];
              const float4 ev = zp[0], od = zp[32];
              const float z8[8] = {ev.x, od.x, ev.y, od.y, ev.z, od.z, ev.w, od.w};
#pragma unroll
              for (int k = 0; k < 8; ++k) g = __builtin_fmaf(v[8 * o + k], z8[k], g);
            }
          }
          __syncthreads();
        }
        run_octets<0, 2>(acc, tile, S, oc, min(end0, oe), zs + lane, rs, lane);
        const int o1 = max(oc, end0);
        run_octets<1, 2>(acc, tile, S, o1, min(end1, oe), zs + (o1 - oc) * 128 + lane, rs, lane);
        __syncthreads();  // the chunk's normals are read; the next may overwrite them
      }
      if (wave == 0) {
        float la = acc.a[1][15], lb = acc.b[1][15];
        swap32(la, lb);  // lb: row 32T - 1 of the lane's path
        sLoss[lane] = loss_row ? -lb : -g;
      }
      uint32_t ca = 0, cb = 0, na = 0, nr = 0;
#pragma unroll
      for (int i = 0; i < kSlots; ++i) {
        if (tile[i] < 0) continue;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const bool excl = r == 15 && h == 1 && i == 1 && wave == 0 && loss_row;
          ca += acc.a[i][r] < a.thr && !excl ? 1u : 0u;
          cb += acc.b[i][r] < a.thr && !excl ? 1u : 0u;
        }
        if (want_near) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const bool excl = r == 15 && h == 1 && i == 1 && wave == 0 && loss_row;
            na |= acc.a[i][r] >= a.thr_lo && acc.a[i][r] <= a.thr_hi && !excl;
            nr |= acc.b[i][r] >= a.thr_lo && acc.b[i][r] <= a.thr_hi && !excl;
          }
        }
      }
      swap32(ca, cb);
      swap32(na, nr);
      sS[wave][lane] = (int)(ca + cb) | ((na | nr) ? (1 << 30) : 0);
      __syncthreads();
      if (wave == 0) {
        int tot = 0, any = 0;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
          const int e = sS[w][lane];
          tot += e & 0xffff;
          any |= e;
        }
        tally_wave(a, &t, q, (uint32_t)(path >> 32) == path_hi && q < a.npaths, tot, sLoss[lane],
                   (any >> 30) & 1, want_hist ? sh_hist : nullptr);
      }
      // sS and sLoss are next written behind the next chunk's barriers
      if (path_hi == (uint32_t)((first + 63) >> 32)) break;
      hi = path_hi + 1;
    }
  }
  __syncthreads();
  flush_tally_lds(a, &t, threadIdx.x);
  if (want_hist) {
    for (int i = threadIdx.x; i <= n; i += blockDim.x)
      if (sh_hist[i]) atomicAdd(&a.s_hist[i], (unsigned long long)sh_hist[i]);
  }
}

// Waves per workgroup and workgroups per CU, four waves per SIMD in all.  The
// normals of 64 paths take n / 4 KiB, so at large n one workgroup fills a CU's LDS
// and has 16 waves; 8 where two fit (n <= 304), 4 where four do (n <= 152), so
// that one's normals run beside another's products and fewer waves meet at a
// barrier: 4e11 / (n^2 + 40 n) paths on 4 against 8 waves n = 143 5.29 / 5.71 ms,
// n = 150 5.00 / 5.50; on 8 against 16 n = 301 4.02 / 4.24.  Two tile slots per
// wave cover T in every case.
F32Shape f32_shape(int n) {
  F32Shape s;
  const int S = (n + 7) / 8;
  s.lds = (size_t)(n <= kMaxN ? S : kChunkCols / 8) * 128 * sizeof(float4) +
          ((n + 1) * sizeof(unsigned) + 15) / 16 * 16;
  // static LDS: counts and losses of 64 paths per wave, the tally
  auto fits = [&](int waves) {
    const size_t stat = sizeof(int) * waves * 64 + sizeof(float) * 64 + sizeof(LdsTally<1>);
    return (int)((160 * 1024) / (s.lds + stat));
  };
  s.waves = fits(4) >= 4 ? 4 : (fits(8) >= 2 ? 8 : 16);
  s.per_cu = 16 / s.waves;  // four waves per SIMD
  s.kernel = s.waves == 16 ? k_f32_lds<16> : (s.waves == 8 ? k_f32_lds<8> : k_f32_lds<4>);
  return s;
}

}  // namespace mcr
