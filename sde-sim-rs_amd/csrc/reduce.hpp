// reduce.hpp -- the compensated f64 reductions across blocks (aot_kernels.hip, basket_kernels.hip,
// batch_kernels.hip). The partials of a run are few (one per block of paths) and on the critical path
// of every evaluation, so what counts is latency: each thread keeps a Neumaier sum of its share,
// with the loads of its iterations independent of the sums, and the sums meet in a butterfly over
// the wave's lanes and then over the waves, log2 steps in a fixed order. (A single thread that
// added the 256 pairs of a block one by one took 24 of the 28 us of a plan's reduction, 2048
// dependent additions.)
#pragma once

#include <hip/hip_runtime.h>

struct SdeSum {
  double s = 0.0, c = 0.0;
  __device__ __forceinline__ void add(double x) {
    const double t = s + x;
    c += (fabs(s) >= fabs(x)) ? (s - t) + x : (x - t) + s;
    s = t;
  }
  __device__ __forceinline__ double value() const { return s + c; }
};

// The sum over the wave's 64 lanes, in every lane.
__device__ __forceinline__ void sde_wave_sum(SdeSum& a) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const double s = __shfl_xor(a.s, off, 64), c = __shfl_xor(a.c, off, 64);
    a.add(s);
    a.c += c;
  }
}

// The sum over the block's threads (whole waves, at most 1024), valid in the first wave. `sh` is
// this reduction's own LDS.
__device__ __forceinline__ void sde_block_sum(SdeSum& a, double (&sh)[16][2]) {
  sde_wave_sum(a);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, waves = blockDim.x >> 6;
  if (lane == 0) {
    sh[wave][0] = a.s;
    sh[wave][1] = a.c;
  }
  __syncthreads();
  if (wave == 0) {
    a = SdeSum();
    if (lane < waves) {
      a.s = sh[lane][0];
      a.c = sh[lane][1];
    }
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) {
      const double s = __shfl_xor(a.s, off, 64), c = __shfl_xor(a.c, off, 64);
      a.add(s);
      a.c += c;
    }
  }
}
