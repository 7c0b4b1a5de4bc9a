// Block sums and sums of block partials for kernels whose blocks are not all kBlock threads.
#pragma once
#include <hip/hip_runtime.h>

#include "device_common.h"

namespace lfric {
namespace {

// sums of several values over a block of NT threads, the same in every thread
template <int NT, int NV>
__device__ inline void block_sum_nt(double (&v)[NV], double (&out)[NV]) {
  __shared__ double sh[NT / 64][NV];
  wave_sum<NV>(v);
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int q = 0; q < NV; ++q) sh[threadIdx.x >> 6][q] = v[q];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) s += sh[w][q];
    out[q] = s;
  }
  __syncthreads();
}

// the sum of nb partials of NV values by a block of NT threads, in one fixed order in every block
template <int NT, int NV>
__device__ inline void sum_partials(const double *__restrict__ p, int nb, double (&tot)[NV]) {
  constexpr int kU = 8;
  double s[NV];
#pragma unroll
  for (int q = 0; q < NV; ++q) s[q] = 0.0;
  for (int b = threadIdx.x; b < nb; b += kU * NT) {
    double t[kU][NV];
#pragma unroll
    for (int u = 0; u < kU; ++u)
#pragma unroll
      for (int q = 0; q < NV; ++q) t[u][q] = b + u * NT < nb ? p[static_cast<size_t>(b + u * NT) * NV + q] : 0.0;
#pragma unroll
    for (int u = 0; u < kU; ++u)
#pragma unroll
      for (int q = 0; q < NV; ++q) s[q] += t[u][q];
  }
  block_sum_nt<NT, NV>(s, tot);
}

}  // namespace
}  // namespace lfric
