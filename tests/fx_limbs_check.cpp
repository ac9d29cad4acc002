// Host driver of the dipole sums' limbs (mtrack_amd/csrc/fixedpoint.h) for
// tests/test_fixedpoint_limbs.py: reads "n block" then n doubles (as 16 hex digits
// of their bits), prints each value's folded limbs as (hi, lo), then the 128-bit
// sum of all of them, accumulated `block` values at a time as a work-group of the
// turn pass does, limbs a stride apart, and its conversion back to double.
#include <stdio.h>
#include <string.h>
#include "fixedpoint.h"

#define STRIDE 5

int main()
{
  long n, block;
  if (scanf("%ld%ld", &n, &block) != 2) return 1;
  unsigned long long slo = 0, shi = 0, acc[FX_LIMBS * STRIDE] = {0};
  unsigned in_block = 0;
  for (long i = 0; i < n; i++) {
    unsigned long long b, l[FX_LIMBS], lo, hi;
    if (scanf("%llx", &b) != 1) return 1;
    double x;
    memcpy(&x, &b, sizeof x);
    fx_limbs(x, l);
    fx_fold(l, 1, 1, lo, hi);
    printf("%016llx %016llx\n", hi, lo);
    for (int k = 0; k < FX_LIMBS; k++) acc[k * STRIDE] += l[k];
    if (++in_block == block || i == n - 1) {
      fx_fold(acc, STRIDE, in_block, lo, hi);
      fx_add(slo, shi, lo, hi);
      memset(acc, 0, sizeof acc);
      in_block = 0;
    }
  }
  const double v = fx_to_double(slo, shi);
  unsigned long long vb;
  memcpy(&vb, &v, sizeof vb);
  printf("sum %016llx %016llx %016llx\n", shi, slo, vb);
  return 0;
}
