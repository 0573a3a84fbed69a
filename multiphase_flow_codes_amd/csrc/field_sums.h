// field_sums.h -- the first level of the global field sums (diag.hip), shared
// by the kernel that reads the rho/u arrays and the one that fills them.
#pragma once
#include <hip/hip_runtime.h>

namespace mfc {

constexpr int kSumThreads = 256;   // threads per reduction block
constexpr int kSumBlocks = 1024, kSumBlocksMax = 4096;   // partial sums of the first level

// Blocks of the first level: one per 2048 nodes within those limits.  More
// blocks fill the memory better, but each leaves six sums to add up: filling
// the arrays and summing took 378 + 5 us at 256^3 FP32 with 1024 blocks, 354 + 8
// with 4096 and 349 + 14 with 8192 (64^3 FP64: 14 + 3.5, 22 + 5.6).
inline int sum_blocks(uint64_t ncell) {
  const uint64_t b = ncell / 2048;
  return (int)(b < kSumBlocks ? kSumBlocks : (b > kSumBlocksMax ? kSumBlocksMax : b));
}

// rho, ux, uy, uz, u.u and the largest u.u over a thread's nodes, i = block *
// kSumThreads + thread and every grid * kSumThreads from there.
struct FieldSums {
  double s[6] = {0, 0, 0, 0, 0, 0};
  __device__ __forceinline__ void add(double rho, double a, double b, double c) {
    const double q = a * a + b * b + c * c;
    s[0] += rho;
    s[1] += a;
    s[2] += b;
    s[3] += c;
    s[4] += q;
    s[5] = fmax(s[5], q);
  }
  // the block's sums to part[6 * block + k] (every thread of the block calls it)
  __device__ __forceinline__ void store(double* __restrict__ part) {
    __shared__ double red[6][kSumThreads / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      double v = s[k];
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        const double t = __shfl_down(v, o, 64);
        v = (k == 5) ? fmax(v, t) : v + t;
      }
      if (lane == 0) red[k][w] = v;
    }
    __syncthreads();
    if (threadIdx.x < 6) {
      const int k = threadIdx.x;
      double v = red[k][0];
      for (int q = 1; q < kSumThreads / 64; ++q) v = (k == 5) ? fmax(v, red[k][q]) : v + red[k][q];
      part[6 * blockIdx.x + k] = v;
    }
  }
};

}  // namespace mfc
