// Expectation values of saved states (used by the DIA integrators).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

namespace dqh {

// expects[inst][k][s] = Tr(E_k rho_s) = sum_ab (E_k^T)_ab (rho_s)_ab over the saved
// states, FP64 accumulation. Bound by reading the states once, so a state is split over
// gridDim.z workgroups whose sums k_expect_sum adds in order (one workgroup per state of
// n = 1024 was bound by the latency of its loads: 1.79 ms for 80 states).
// grid: (nsave, ninst, chunks); block 256. part: [ninst][nsave][nE][chunks], unused with
// one chunk.
static __global__ __launch_bounds__(256) void k_expect_states(int64_t n_true, int64_t nsave, int64_t nE,
                                                const float2 *__restrict__ states, const float2 *__restrict__ EopsT,
                                                float2 *__restrict__ expects, double2 *__restrict__ part) {
  __shared__ double red[4][2];
  const int64_t s = blockIdx.x;
  const size_t inst = blockIdx.y, chunks = gridDim.z;
  const size_t nn = (size_t)n_true * n_true;
  const size_t len = (nn + chunks - 1) / chunks, e0 = blockIdx.z * len, e1 = e0 + len < nn ? e0 + len : nn;
  const float2 *R = states + (inst * nsave + s) * nn;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int64_t k = 0; k < nE; ++k) {
    const float2 *Ek = EopsT + k * nn;
    double ar = 0.0, ai = 0.0;
#pragma unroll 4
    for (size_t e = e0 + threadIdx.x; e < e1; e += 256) {
      const float2 a = Ek[e], r = R[e];
      ar += (double)a.x * r.x - (double)a.y * r.y;
      ai += (double)a.x * r.y + (double)a.y * r.x;
    }
    for (int o = 32; o > 0; o >>= 1) {
      ar += __shfl_xor(ar, o, 64);
      ai += __shfl_xor(ai, o, 64);
    }
    __syncthreads();
    if (lane == 0) {
      red[wave][0] = ar;
      red[wave][1] = ai;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      double sr = 0.0, si = 0.0;
      for (int w = 0; w < 4; ++w) {
        sr += red[w][0];
        si += red[w][1];
      }
      if (chunks == 1)
        expects[(inst * nE + k) * nsave + s] = make_float2((float)sr, (float)si);
      else
        part[((inst * nsave + s) * nE + k) * chunks + blockIdx.z] = make_double2(sr, si);
    }
  }
}

static __global__ __launch_bounds__(256) void k_expect_sum(int64_t nsave, int64_t nE, int64_t count, int chunks,
                                                           const double2 *__restrict__ part, float2 *__restrict__ expects) {
  const int64_t o = (int64_t)blockIdx.x * 256 + threadIdx.x;  // (inst * nsave + s) * nE + k
  if (o >= count) return;
  double sr = 0.0, si = 0.0;
  for (int z = 0; z < chunks; ++z) {
    const double2 x = part[o * chunks + z];
    sr += x.x;
    si += x.y;
  }
  const int64_t k = o % nE, is = o / nE, s = is % nsave, inst = is / nsave;
  expects[(inst * nE + k) * nsave + s] = make_float2((float)sr, (float)si);
}

// nsave, ninst, nE >= 1; scratch: device memory that is free by then
static inline void launch_expect(int64_t n_true, int64_t nsave, int64_t ninst, int64_t nE, uint64_t states,
                                 uint64_t EopsT, uint64_t expects, void *scratch, size_t bytes, hipStream_t st) {
  const int64_t count = ninst * nsave * nE, fit = (int64_t)(bytes / sizeof(double2)) / count;
  // from 8192 elements per workgroup (32 per thread) the sums hide their latency
  const int64_t chunks = std::max<int64_t>(1, std::min<int64_t>({fit, 64, n_true * n_true / 8192}));
  float2 *ex = reinterpret_cast<float2 *>(expects);
  double2 *part = reinterpret_cast<double2 *>(scratch);
  hipLaunchKernelGGL(k_expect_states, dim3((unsigned)nsave, (unsigned)ninst, (unsigned)chunks), dim3(256), 0, st, n_true,
                     nsave, nE, reinterpret_cast<const float2 *>(states), reinterpret_cast<const float2 *>(EopsT), ex, part);
  if (chunks > 1)
    hipLaunchKernelGGL(k_expect_sum, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, st, nsave, nE, count, (int)chunks,
                       part, ex);
}

}  // namespace dqh
