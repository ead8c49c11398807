// mcr_rng.h -- the counter-based normal stream every kernel draws from.
//
// Replaces the per-thread cuRAND XORWOW state of the reference GPU model
// (src/05-GPU/monte_carlos_cuda.cu:30-31 curand_init(seed, idx, 0) and :45-47
// curand_normal_double) and the sequential GSL MT19937 stream of the CPU models
// (src/02-C-serial/monte_carlo_serial.c:46,54,67-69).  Nothing of cuRAND is
// reproduced: the generator is Philox4x32-10 as published by Salmon, Moraes,
// Dror and Shaw, "Parallel Random Numbers: As Easy as 1, 2, 3" (SC'11), and the
// normal transform is Box-Muller with this file's own polynomial kernels.
//
// Stream definition (the contract a host mirror must follow bit for bit):
//   key     = (seed & 0xffffffff, seed >> 32)
//   counter = (block, 0, path & 0xffffffff, path >> 32)
//   (x0,x1,x2,x3) = Philox4x32-10(counter, key)
//   z[4*block+0], z[4*block+1] = BoxMuller(x0, x1)
//   z[4*block+2], z[4*block+3] = BoxMuller(x2, x3)
//   BoxMuller(a, b):  u = ((a >> 8) + 1) * 2^-24  in [2^-24, 1]
//                     r = sqrt(-2 ln u),   theta = 2*pi * b / 2^32
//                     (r cos theta, r sin theta)
// Every step uses only integer ops and IEEE fp32 add/mul/fma (no libm, no
// hardware transcendental), so a host compiled with fp contraction off
// reproduces each normal exactly.  Must be compiled with -ffp-contract=off.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#define MCR_HD __host__ __device__ __forceinline__
#else
#define MCR_HD static inline
#endif

namespace mcr {

// Philox4x32 round constants (Salmon et al. SC'11, Table 2 / Random123).
constexpr uint32_t kPhiloxM0 = 0xD2511F53u;
constexpr uint32_t kPhiloxM1 = 0xCD9E8D57u;
constexpr uint32_t kPhiloxW0 = 0x9E3779B9u;  // golden ratio
constexpr uint32_t kPhiloxW1 = 0xBB67AE85u;  // sqrt(3) - 1

struct Ctr4 {
  uint32_t x, y, z, w;
};

// a ^ b ^ c in one v_bitop3_b32 on gfx950 (truth table 0x96); plain xors on the host
MCR_HD uint32_t xor3(uint32_t a, uint32_t b, uint32_t c) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);
#else
  return a ^ b ^ c;
#endif
}

struct Key2 {
  uint32_t k0, k1;
};
MCR_HD Key2 key_of(uint64_t seed) { return Key2{(uint32_t)seed, (uint32_t)(seed >> 32)}; }

// Rounds R0 .. 9 of the ten.
template <int R0>
MCR_HD Ctr4 philox_rounds(Ctr4 c, Key2 k) {
  uint32_t k0 = k.k0 + R0 * kPhiloxW0, k1 = k.k1 + R0 * kPhiloxW1;
#pragma unroll
  for (int r = R0; r < 10; ++r) {
    const uint64_t p0 = (uint64_t)kPhiloxM0 * c.x;
    const uint64_t p1 = (uint64_t)kPhiloxM1 * c.z;
    c = Ctr4{xor3((uint32_t)(p1 >> 32), c.y, k0), (uint32_t)p1, xor3((uint32_t)(p0 >> 32), c.w, k1),
             (uint32_t)p0};
    k0 += kPhiloxW0;
    k1 += kPhiloxW1;
  }
  return c;
}
MCR_HD Ctr4 philox4x32_10(Ctr4 c, uint32_t k0, uint32_t k1) {
  return philox_rounds<0>(c, Key2{k0, k1});
}

// Counter (block, 0, path lo, path hi): the first two of the ten rounds hold
// products of the path's low word alone (once per path) and products of the
// block and the path's high word alone.  Kernels whose block index and path
// high word are uniform over a wave get the latter from the scalar unit, which
// leaves 16 of the 20 64-bit products of a block to the vector unit.
struct PhiloxPath {
  uint32_t y1;      // round 1: y
  uint32_t zh, w2;  // round 2: z before the block's part, w
};
struct PhiloxBlock {
  uint32_t x2, y2, zb;  // round 2: x before the path's part, y, the block's part of z
};

MCR_HD PhiloxPath philox_path(uint32_t path_lo, Key2 k) {
  const uint64_t p1 = (uint64_t)kPhiloxM1 * path_lo;
  const uint64_t p0 = (uint64_t)kPhiloxM0 * ((uint32_t)(p1 >> 32) ^ k.k0);
  return PhiloxPath{(uint32_t)p1, (uint32_t)(p0 >> 32), (uint32_t)p0};
}

MCR_HD PhiloxBlock philox_block(uint32_t blk, uint32_t path_hi, Key2 k) {
  const uint64_t p0 = (uint64_t)kPhiloxM0 * blk;
  const uint64_t p1 = (uint64_t)kPhiloxM1 * ((uint32_t)(p0 >> 32) ^ path_hi ^ k.k1);
  return PhiloxBlock{(uint32_t)(p1 >> 32) ^ (k.k0 + kPhiloxW0), (uint32_t)p1,
                     (uint32_t)p0 ^ (k.k1 + kPhiloxW1)};
}

MCR_HD Ctr4 philox4x32_10(PhiloxPath p, PhiloxBlock b, Key2 k) {
  return philox_rounds<2>(Ctr4{p.y1 ^ b.x2, b.y2, p.zh ^ b.zb, p.w2}, k);
}

MCR_HD float as_f32(uint32_t b) { return __builtin_bit_cast(float, b); }
MCR_HD uint32_t as_u32(float f) { return __builtin_bit_cast(uint32_t, f); }

// Near-minimax coefficients (Lawson-reweighted least squares on Chebyshev
// nodes, rounded to fp32; the fit script is derive_normal_poly.py beside this
// file).  ln(1+f) = f - f^2/2 + f^3 P(f) on f in [sqrt(1/2)-1, sqrt(2)-1],
// max relative error 3.5e-8.
constexpr float kLogP0 = 0x1.5556d8p-2f;
constexpr float kLogP1 = -0x1.000382p-2f;
constexpr float kLogP2 = 0x1.98d7f0p-3f;
constexpr float kLogP3 = -0x1.53824cp-3f;
constexpr float kLogP4 = 0x1.31747cp-3f;
constexpr float kLogP5 = -0x1.2432a4p-3f;
constexpr float kLogP6 = 0x1.645d88p-4f;
constexpr float kLn2Hi = 0x1.62e400p-1f;  // 16 significant bits: e*kLn2Hi exact
constexpr float kLn2Lo = 0x1.7f7d1cp-20f;
// sin(2 pi a) = a S(a^2), cos(2 pi a) = 1 + a^2 C(a^2) on a in [-1/8, 1/8]
// (turns); max relative error 3.6e-8 (sin), absolute 6.7e-9 (cos).
constexpr float kSin0 = 0x1.921fb6p+2f;
constexpr float kSin1 = -0x1.4abbbap+5f;
constexpr float kSin2 = 0x1.465ec8p+6f;
constexpr float kSin3 = -0x1.2d9bf2p+6f;
constexpr float kCos1 = -0x1.3bd3ccp+4f;
constexpr float kCos2 = 0x1.03c1dep+6f;
constexpr float kCos3 = -0x1.55c664p+6f;
constexpr float kCos4 = 0x1.d9f7bep+5f;

// The transform below computes the stream definition's r and theta with as few
// instructions as give the same bits (a Box-Muller pair takes 49 VALU
// instructions against 56 for the plain form; checked on the host over all
// 2^24 logarithm inputs and all 2^32 angles.  With the packed bf16 conversion
// of the path kernels a query of n = 50, 1e8 paths went from 5.71 to 5.11 ms):
//  - the exponent of u stays in place, as e * 2^23, so that subtracting it from
//    the bit pattern gives the mantissa and converting it gives e scaled by a
//    power of two, which the ln 2 constants take back;
//  - the logarithm keeps its sign (l = ln u <= 0): the root reads -l = h through
//    its seed constant and the sign of its Newton product;
//  - the root's factor 2 sits in the sine and cosine coefficients (powers of
//    two commute with rounding);
//  - the quarter turn's sign goes onto the radius, once for both results, and
//    its parity is read as a float compare.

// ln(u) for u = ((a >> 8) + 1) * 2^-24.  Range reduction u = 2^e m with
// m in [sqrt(1/2), sqrt(2)) done on the fp32 bit pattern.
MCR_HD float log_u24(uint32_t a) {
  const float u = __builtin_fmaf((float)(a >> 8), 0x1p-24f, 0x1p-24f);  // exact
  const uint32_t ub = as_u32(u);
  const uint32_t eh = (ub - 0x3f3504f3u) & 0xff800000u;  // e * 2^23
  const float f = as_f32(ub - eh) - 1.0f;                // m - 1, exact (Sterbenz)
  float p = kLogP6;
  p = __builtin_fmaf(p, f, kLogP5);
  p = __builtin_fmaf(p, f, kLogP4);
  p = __builtin_fmaf(p, f, kLogP3);
  p = __builtin_fmaf(p, f, kLogP2);
  p = __builtin_fmaf(p, f, kLogP1);
  p = __builtin_fmaf(p, f, kLogP0);
  const float q = __builtin_fmaf(p, f, -0.5f);
  const float t = f * f;
  const float l1p = __builtin_fmaf(t, q, f);
  const float ef = (float)(int32_t)eh;
  const float lo = __builtin_fmaf(ef, kLn2Lo * 0x1p-23f, l1p);
  return __builtin_fmaf(ef, kLn2Hi * 0x1p-23f, lo);
}

// sqrt(2 h) / 2 for l = -h, h in [0, 17]: bit-pattern seed for 1/sqrt(2h)
// (Lomont's constant 0x5f375a86 with the factor 2 folded into the exponent and
// the sign bit of l, which the shift brings down, taken out; 3.4% worst error),
// three Newton steps g <- g (3/2 - h g^2) (error 1.7e-3, 4.6e-6, then fp32
// rounding), then h * g.  At h = 0 (l = +0) the seed is a tiny negative number,
// the iteration keeps it finite and the result is -0.
MCR_HD float half_sqrt_twice(float l) {
  float g = as_f32(0x9ef75a86u - (as_u32(l) >> 1));
#pragma unroll
  for (int it = 0; it < 3; ++it) {
    float t = g * g;
    t = __builtin_fmaf(l, t, 1.5f);
    g = g * t;
  }
  return __builtin_fabsf(l) * g;
}

// (r cos theta, r sin theta) for theta = 2 pi b / 2^32 and hr = r / 2.  The
// nearest quarter turn q comes from the top bits of b, the signed remainder (30
// bits) is the reduced argument in turns; s and c below are twice its sine and
// cosine.
MCR_HD void rotate_turn(uint32_t b, float hr, float* z0, float* z1) {
  const int32_t rem = (int32_t)(b << 2) >> 2;
  uint32_t q = b - (uint32_t)rem;  // quarter turns, in bits 30 and 31
#if defined(__HIP_DEVICE_COMPILE__)
  // opaque, or the compare below becomes a mask and an integer compare
  asm("" : "+v"(q));
#endif
  const float a = (float)rem * 0x1p-32f;
  const float t = a * a;
  float s = __builtin_fmaf(2.0f * kSin3, t, 2.0f * kSin2);
  s = __builtin_fmaf(s, t, 2.0f * kSin1);
  s = __builtin_fmaf(s, t, 2.0f * kSin0);
  s = s * a;
  float c = __builtin_fmaf(2.0f * kCos4, t, 2.0f * kCos3);
  c = __builtin_fmaf(c, t, 2.0f * kCos2);
  c = __builtin_fmaf(c, t, 2.0f * kCos1);
  c = __builtin_fmaf(c, t, 2.0f);
  const float w = as_f32(as_u32(hr) ^ (q & 0x80000000u));
  const bool odd = as_f32(q) != 0.0f;  // 2.0 or -2.0, against 0.0 and -0.0
  *z0 = w * (odd ? -s : c);
  *z1 = w * (odd ? c : s);
}

MCR_HD void box_muller(uint32_t a, uint32_t b, float* z0, float* z1) {
  rotate_turn(b, half_sqrt_twice(log_u24(a)), z0, z1);
}

// Normals z[4*blk .. 4*blk+3] of one path.
MCR_HD void normals4(Key2 key, PhiloxPath path, PhiloxBlock blk, float z[4]) {
  const Ctr4 x = philox4x32_10(path, blk, key);
  box_muller(x.x, x.y, &z[0], &z[1]);
  box_muller(x.z, x.w, &z[2], &z[3]);
}
MCR_HD void normals4(Key2 key, uint64_t path, uint32_t blk, float z[4]) {
  normals4(key, philox_path((uint32_t)path, key), philox_block(blk, (uint32_t)(path >> 32), key), z);
}

// normals4's z[0], z[1] alone (the same bits): for a path's last block when
// n leaves its second pair unused.
MCR_HD void normals2(Key2 key, PhiloxPath path, PhiloxBlock blk, float z[2]) {
  const Ctr4 x = philox4x32_10(path, blk, key);
  box_muller(x.x, x.y, &z[0], &z[1]);
}
MCR_HD void normals2(Key2 key, uint64_t path, uint32_t blk, float z[2]) {
  normals2(key, philox_path((uint32_t)path, key), philox_block(blk, (uint32_t)(path >> 32), key), z);
}

}  // namespace mcr
