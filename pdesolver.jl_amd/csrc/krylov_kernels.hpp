// krylov_kernels.hpp -- sums shared by the single and the batched GMRES kernels.
#pragma once
#include "pdes_common.hpp"

namespace pdes {

constexpr int CGS_THREADS = 256;
// rows of at most this many partial sums are added up by every workgroup that
// needs them; longer ones once, in a launch of its own
constexpr int CGS_SELF_REDUCE = 256;

__device__ __forceinline__ double wave_sum(double x) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
  return x;
}

// Sums of NV values over the lanes of a wave, NV a power of two up to 64: each
// exchange halves the values a lane keeps, so NV - 1 of them serve all.  Lane
// l ends with the sum of value l / (64 / NV).
template <int NV, int HALF = NV / 2, int OFF = 32>
__device__ __forceinline__ double wave_sums(double (&v)[NV]) {
  if constexpr (OFF == 0) {
    return v[0];
  } else if constexpr (HALF == 0) {
    v[0] += __shfl_xor(v[0], OFF, 64);
    return wave_sums<NV, 0, OFF / 2>(v);
  } else {
    const bool up = threadIdx.x & OFF;
#pragma unroll
    for (int k = 0; k < HALF; ++k) {
      const double give = up ? v[k] : v[k + HALF], keep = up ? v[k + HALF] : v[k];
      v[k] = keep + __shfl_xor(give, OFF, 64);
    }
    return wave_sums<NV, HALF / 2, OFF / 2>(v);
  }
}

// h[i] = sum of partial[i * ld + b] over b < nb <= CGS_SELF_REDUCE, i < m: each
// wave of the workgroup sums 8 rows at a time
__device__ __forceinline__ void sum_partial_rows(const double* __restrict__ partial, int m, int nb, int64_t ld,
                                                 double* h) {
  const int lane = threadIdx.x & 63;
  for (int i0 = 8 * (threadIdx.x >> 6); i0 < m; i0 += 8 * (CGS_THREADS / 64)) {
    double x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = 0.0;
    // (all of a wave's loads in flight together)
    double v[8][CGS_SELF_REDUCE / 64];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int k = 0; k < CGS_SELF_REDUCE / 64; ++k) {
        const int b = lane + 64 * k;
        v[i][k] = i0 + i < m && b < nb ? partial[(int64_t)(i0 + i) * ld + b] : 0.0;
      }
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int k = 0; k < CGS_SELF_REDUCE / 64; ++k) x[i] += v[i][k];
    const double y = wave_sums<8>(x);
    if (lane % 8 == 0 && i0 + lane / 8 < m) h[i0 + lane / 8] = y;
  }
  __syncthreads();
}

}  // namespace pdes
