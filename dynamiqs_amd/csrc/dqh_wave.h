// Wave and workgroup sums, and the tableau in scalar registers, for the persistent kernels
// that keep their stages in registers (gfx950).
#pragma once

#include <hip/hip_runtime.h>

#include "dqh_tsit5_tableau.h"

namespace dqh {

// x + (x of the lane that the DPP control names)
template <int CTRL>
__device__ __forceinline__ double dpp_sum(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
  return x + __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double lane_of(double x, int lane) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_readlane((int)b, lane), hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// sum over the wave, the same value in every lane: butterfly over quads, half rows and
// rows of 16 lanes on the VALU, then the four rows through scalar registers
__device__ __forceinline__ double wave_sum(double x) {
  x = dpp_sum<0xB1>(x);   // lane ^ 1
  x = dpp_sum<0x4E>(x);   // lane ^ 2
  x = dpp_sum<0x141>(x);  // the other quad of the half row
  x = dpp_sum<0x140>(x);  // the other half of the row
  return (lane_of(x, 0) + lane_of(x, 16)) + (lane_of(x, 32) + lane_of(x, 48));
}

// sum over the quad of lanes, alike in all four
__device__ __forceinline__ float quad_sum(float x) {
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0xB1, 0xf, 0xf, true));
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x4E, 0xf, 0xf, true));
  return x;
}

// workgroup sums of N values with one barrier; red alternates between two halves, so a
// second call need not wait for the readers of the first
template <int NTH, int N>
__device__ __forceinline__ void block_sums(double (&x)[N], double *red, int &par) {
  constexpr int NW = NTH / 64;
#pragma unroll
  for (int k = 0; k < N; ++k) x[k] = wave_sum(x[k]);
  double *r = red + par * (NW * 2);
  par ^= 1;
  if constexpr (NW > 1) {
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
      for (int k = 0; k < N; ++k) r[2 * (threadIdx.x >> 6) + k] = x[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < N; ++k) {
      double s = 0.0;
#pragma unroll
      for (int w = 0; w < NW; ++w) s += r[2 * w + k];
      x[k] = s;
    }
  }
}

// the tableau through a scalar pointer that the optimiser cannot see through: its loads
// stay where they are used (as literals, or hoisted out of the loop, the weights would
// fill the registers that the stages need)
typedef const __attribute__((address_space(4))) RKTab CTab;
template <int TAB>
__device__ __forceinline__ CTab *weights() {
  CTab *r = (CTab *)&kRK[TAB];
  asm volatile("" : "+s"(r));
  return r;
}

}  // namespace dqh
