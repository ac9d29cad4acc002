// Exact 128-bit fixed point of the slice dipole sums: a double x, |x| < 2^20,
// becomes the two's-complement integer round(x 2^100), a sum of such integers held
// in two 64-bit words (lo, hi); sums are exact and independent of their order while
// their magnitude stays below 2^27.  k_turn forms the integer as three limbs
// (fx_limbs, ties to even) and folds a block's limb sums into the two words
// (fx_fold); fx_split forms the words of one value at once (ties away from zero,
// so that the two differ by one unit of 2^-100 exactly at ties) and serves the unit
// tests as the plain form.
// Host and device code (the host side serves the unit tests of these helpers).
#ifndef MBT_FIXEDPOINT_H
#define MBT_FIXEDPOINT_H
#include <hip/hip_runtime.h>
#include <math.h>
#include <string.h>

__host__ __device__ inline void fx_split(double x, unsigned long long &lo, unsigned long long &hi)
{
  unsigned long long bits;
  memcpy(&bits, &x, sizeof bits);
  const int e = (int)((bits >> 52) & 0x7ff);
  const unsigned long long m = (bits & 0xfffffffffffffULL) | (1ULL << 52);
  lo = 0;
  hi = 0;
  if (e == 0) return;
  const int s = e - 975; // x 2^100 = m 2^s
  if (s >= 64) {
    hi = m << (s - 64);
  } else if (s > 0) {
    lo = m << s;
    hi = m >> (64 - s);
  } else if (s == 0) {
    lo = m;
  } else if (s > -64) {
    const int r = -s;
    lo = (m >> r) + ((m >> (r - 1)) & 1ULL);
  } else if (s == -64) {
    lo = (m >> 63) & 1ULL;
  }
  if (bits >> 63) { // negate
    lo = ~lo + 1ULL;
    hi = ~hi + (lo == 0ULL ? 1ULL : 0ULL);
  }
}

// (lo, hi) += (a, b), modulo 2^128
__host__ __device__ inline void fx_add(unsigned long long &lo, unsigned long long &hi, unsigned long long a,
                                       unsigned long long b)
{
  const unsigned long long old = lo;
  lo += a;
  hi += b + (lo < old ? 1ULL : 0ULL);
}

// The block's dipole sums in LDS: x = A 2^-20 + B 2^-60 + C 2^-100 with A, B, C
// integers, |A| <= 2^40, |B| and |C| <= 2^39, each added to a 64-bit accumulator of its
// slice.  A limb is rounded (to nearest, ties to even) by adding 1.5 2^52, whose
// bits then hold the integer in their low half; what is left over is exact, so
// only C's rounding loses anything.  The bits are added as they are and FX_MAGIC
// times the number of values taken off when the block's sums are folded.  Adding
// the two words instead needed the old value of every addition for the carry, and
// shifts by the exponent's range with a branch each: 143 instructions a
// macroparticle and two waits for LDS, now 24 and none.
#define FX_LIMBS 3
#define FX_MAGIC_D 6755399441055744.0 // 1.5 2^52
#define FX_MAGIC 0x4338000000000000ULL

__host__ __device__ inline unsigned long long fx_bits(double v)
{
  unsigned long long b;
  memcpy(&b, &v, sizeof b);
  return b;
}

__host__ __device__ inline void fx_limbs(double x, unsigned long long l[FX_LIMBS])
{
  const double u = 1048576.0, w = 1099511627776.0; // 2^20, 2^40
  const double a = fma(x, u, FX_MAGIC_D);
  double r = fma(x, u, FX_MAGIC_D - a);
  const double b = fma(r, w, FX_MAGIC_D);
  r = fma(r, w, FX_MAGIC_D - b);
  const double c = fma(r, w, FX_MAGIC_D);
  l[0] = fx_bits(a);
  l[1] = fx_bits(b);
  l[2] = fx_bits(c);
}

// the accumulated limbs of n values (stride apart) as the 128-bit sum (lo, hi)
__host__ __device__ inline void fx_fold(const unsigned long long *l, int stride, unsigned n, unsigned long long &lo,
                                        unsigned long long &hi)
{
  const long long a = (long long)(l[0] - n * FX_MAGIC), b = (long long)(l[stride] - n * FX_MAGIC),
                  c = (long long)(l[2 * stride] - n * FX_MAGIC);
  lo = (unsigned long long)c;
  hi = (unsigned long long)(c >> 63);
  fx_add(lo, hi, (unsigned long long)b << 40, (unsigned long long)(b >> 24));
  hi += (unsigned long long)a << 16;
}

__host__ __device__ inline double fx_to_double(unsigned long long lo, unsigned long long hi)
{
  const long long h = (long long)hi;
  const double v = (double)h * 18446744073709551616.0 + (double)lo;
  return v * 7.888609052210118e-31; // 2^-100
}
#endif
