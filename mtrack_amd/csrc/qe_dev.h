// Normals of the quantum excitation, device code of the turn pass.
#ifndef MBT_QE_DEV_H
#define MBT_QE_DEV_H
#include <hip/hip_runtime.h>
#include <stdint.h>

#pragma clang fp contract(off)

// Philox4x32-10 and the QE normals: the oracle's orc_qe_normals (float Box-Muller
// from explicit-FMA polynomials) bit for bit.  With quantum excitation the turn
// is VALU-bound, so each step is the fewest instructions that give the same
// bits (checked over all 2^24 inputs of both Box-Muller functions): the product
// of a Philox round as one v_mad_u64_u32, its three-way xor as one v_bitop3_b32,
// no scaling of operands that cannot leave the normal range, no branches.  The
// loop of k_turn with excitation went from 730 vector instructions a
// macroparticle to 600 (with dipole histograms too from 790 to 615; see the note
// at its loops for the time).
__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c)
{
  return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);
}

__device__ __forceinline__ void philox(uint32_t c[4], uint32_t k0, uint32_t k1)
{
#pragma unroll
  for (int r = 0; r < 10; r++) {
    const uint64_t p0 = (uint64_t)0xD2511F53u * c[0], p1 = (uint64_t)0xCD9E8D57u * c[2];
    const uint32_t n0 = xor3((uint32_t)(p1 >> 32), c[1], k0), n2 = xor3((uint32_t)(p0 >> 32), c[3], k1);
    c[0] = n0;
    c[1] = (uint32_t)p1;
    c[2] = n2;
    c[3] = (uint32_t)p0;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
}

// sqrt(-2 ln u), u = ((x >> 8) + 1) / 2^24 in (0, 1].  ln u from u = 2^e m, m in
// [0.70710677, 1.4142135], as 2 atanh(s), s = (m - 1) / (m + 1).
__device__ __forceinline__ float qe_radius(uint32_t x)
{
  // subtracting the bits of 2^24 0.70710677 leaves e in the exponent field
  const uint32_t ix = __float_as_uint((float)((x >> 8) + 1u)) - (0x3f3504f4u + (24u << 23));
  const float e = (float)((int)ix >> 23), m = __uint_as_float((ix & 0x007fffffu) + 0x3f3504f4u);
  // the quotient rounded to nearest: a reciprocal improved by one Newton step, the
  // quotient by its exact remainder (Markstein, IBM J. Res. Dev. 34 (1990) 111)
  const float n = m - 1.0f, d = m + 1.0f;
  float y = __builtin_amdgcn_rcpf(d);
  y = fmaf(fmaf(-d, y, 1.0f), y, y);
  float s = n * y;
  s = fmaf(fmaf(-d, s, n), y, s);
  const float s2 = s * s;
  float p = fmaf(s2, 0.11111111f, 0.14285715f);
  p = fmaf(s2, p, 0.2f);
  p = fmaf(s2, p, 0.33333334f);
  p = fmaf(s2, p, 1.0f);
  const float v = -2.0f * fmaf(e, 0.69314718f, 2.0f * s * p);
  // the square root rounded to nearest: the hardware's, within one unit in the
  // last place, or its neighbour, by the sign of the exact residuals
  const float g = __builtin_amdgcn_sqrtf(v);
  const float lo = __uint_as_float(__float_as_uint(g) - 1u), hi = __uint_as_float(__float_as_uint(g) + 1u);
  float r = fmaf(-lo, g, v) <= 0.0f ? lo : g;
  r = fmaf(-hi, g, v) > 0.0f ? hi : r;
  return r;
}

// sin and cos of 2 pi u, u as above: u = q / 4 + r exactly, |r| <= 1 / 8
__device__ __forceinline__ void qe_sincos(uint32_t b, float *s, float *c)
{
  const float k = (float)((b >> 8) + 1u);
  const float q = rintf(k * 2.3841858e-7f); // k / 2^22
  const float x = fmaf(q, -4194304.0f, k) * (6.2831855f * 5.9604645e-8f);
  const float x2 = x * x;
  float sp = fmaf(x2, 2.7557319e-6f, -1.9841270e-4f);
  sp = fmaf(x2, sp, 8.3333333e-3f);
  sp = fmaf(x2, sp, -0.16666667f);
  const float sn = fmaf(x * x2, sp, x);
  float cp = fmaf(x2, 2.4801587e-5f, -1.3888889e-3f);
  cp = fmaf(x2, cp, 4.1666667e-2f);
  cp = fmaf(x2, cp, -0.5f);
  const float cs = fmaf(x2, cp, 1.0f);
  // quadrant q mod 4: swap on odd, sin negative for 2 and 3, cos for 1 and 2
  const uint32_t iq = (uint32_t)(int)q;
  const bool odd = iq & 1u;
  const uint32_t sb = __float_as_uint(odd ? cs : sn), cb = __float_as_uint(odd ? sn : cs);
  *s = __uint_as_float(__builtin_amdgcn_bitop3_b32(sb, iq << 30, 0x80000000u, 0x78));        // sb ^ (bit 1 of q)
  *c = __uint_as_float(__builtin_amdgcn_bitop3_b32(cb, (iq + 1u) << 30, 0x80000000u, 0x78));
}

__device__ __forceinline__ void bm_pair(uint32_t a, uint32_t b, double &n0, double &n1)
{
  const float r = qe_radius(a);
  float s, c;
  qe_sincos(b, &s, &c);
  n0 = (double)(r * c);
  n1 = (double)(r * s);
}

__device__ __forceinline__ void qe_normals(uint32_t seed, uint32_t bucket, unsigned long long rev, uint32_t j, double n[5])
{
  uint32_t c[4] = {j, (uint32_t)rev, (uint32_t)(rev >> 32), 0u};
  philox(c, seed, bucket);
  bm_pair(c[0], c[1], n[0], n[1]);
  bm_pair(c[2], c[3], n[2], n[3]);
  uint32_t d[4] = {j, (uint32_t)rev, (uint32_t)(rev >> 32), 1u};
  philox(d, seed, bucket);
  double t;
  bm_pair(d[0], d[1], n[4], t);
}

#endif
