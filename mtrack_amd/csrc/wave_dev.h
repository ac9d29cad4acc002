// Sums over the 64 lanes of a wave (gfx950) by DPP moves and half-wave swaps.
#ifndef MBT_WAVE_DEV_H
#define MBT_WAVE_DEV_H
#include <hip/hip_runtime.h>

// A double from another lane of the same row of 16 by a DPP move (no LDS
// permute): CTRL 0x140 = row_mirror (lane 15 - i), 0x141 = row_half_mirror
// (lane 7 - i within each 8), 0x4E = quad_perm [2,3,0,1], 0xB1 = quad_perm
// [1,0,3,2].  Every partner is an involution, so both lanes of a pair form the
// same sum and a butterfly over these four steps leaves the same total in all
// 16 lanes, as the xor butterfly does.  Every partner is a lane of the row, so
// bound_ctrl changes no value; it spares the move of the unused old operand.
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v)
{
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xF, 0xF, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Sum over the row of 16 lanes, in every lane of the row.
__device__ __forceinline__ double rowsum16(double v)
{
  v += dpp_d<0x140>(v);
  v += dpp_d<0x141>(v);
  v += dpp_d<0x4E>(v);
  v += dpp_d<0xB1>(v);
  return v;
}

__device__ __forceinline__ double wsum64(double v)
{
  v += __shfl_xor(v, 32, 64);
  v += __shfl_xor(v, 16, 64);
  return rowsum16(v);
}

// One halving exchange over lane distance D = 32 or 16 without selects: lanes
// with bit D clear return a + (a of the lane D up), lanes with it set (b of the
// lane D down) + b.  v_permlane32_swap exchanges lanes 32-63 of its first
// operand with lanes 0-31 of its second, v_permlane16_swap the odd rows of 16
// of the first with the even rows of the second; one per 32-bit half.
template <int D>
__device__ __forceinline__ double swap_sum(double a, double b)
{
  const unsigned long long ia = (unsigned long long)__double_as_longlong(a);
  const unsigned long long ib = (unsigned long long)__double_as_longlong(b);
  unsigned lo0, lo1, hi0, hi1;
  if (D == 32) {
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)ia, (unsigned)ib, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(ia >> 32), (unsigned)(ib >> 32), false, false);
    lo0 = lo[0], lo1 = lo[1], hi0 = hi[0], hi1 = hi[1];
  } else {
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)ia, (unsigned)ib, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(ia >> 32), (unsigned)(ib >> 32), false, false);
    lo0 = lo[0], lo1 = lo[1], hi0 = hi[0], hi1 = hi[1];
  }
  const double x = __longlong_as_double((long long)(((unsigned long long)hi0 << 32) | lo0));
  const double y = __longlong_as_double((long long)(((unsigned long long)hi1 << 32) | lo1));
  return x + y;
}

// Eight sums over the 64 lanes of a wave at once: three halving exchanges (xor
// 32, 16, 8) split the eight values between lane groups, three more (xor 4, 2,
// 1) finish each; lanes 8k .. 8k+7 return the total of v[k].  Ten exchanges
// instead of 48 for eight separate reductions; a fixed tree, so reproducible.
__device__ __forceinline__ double wsum64x8(const double v[8])
{
  const bool b3 = threadIdx.x & 8;
  double w[4], x[2];
#pragma unroll
  for (int k = 0; k < 4; k++) w[k] = swap_sum<32>(v[k], v[4 + k]);
#pragma unroll
  for (int k = 0; k < 2; k++) x[k] = swap_sum<16>(w[k], w[2 + k]);
  // bit 3 by the row mirror (its partner 15 - i has bit 3 flipped), then the
  // remaining three bits within each half row
  double y = (b3 ? x[1] : x[0]) + dpp_d<0x140>(b3 ? x[0] : x[1]);
  y += dpp_d<0x141>(y);
  y += dpp_d<0x4E>(y);
  y += dpp_d<0xB1>(y);
  return y;
}

// Two sums over the 64 lanes of a wave: lanes 0-31 return the total of a, lanes
// 32-63 that of b.
__device__ __forceinline__ double wsum64x2(double a, double b)
{
  const double x = swap_sum<32>(a, b);
  return rowsum16(swap_sum<16>(x, x));
}

#endif
