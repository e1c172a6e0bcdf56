// batch_kernels.hip -- many independent 1-D SDE instances of uneven size in one launch.
//
// Built-in models with run-time parameters (their DSL forms, compiled by the generic path, give
// bit-identical f64 paths):
//   GBM  dX = (mu * X) * dt + (sigma * X) * dW1
//   OU   dX = (kappa * (theta - X)) * dt + (sigma) * dW1
//   CIR  dX = (kappa * (theta - max(X, 0))) * dt + (sigma * max(X, 0)^0.5) * dW1
// Euler-Maruyama (src/sim/euler.rs:5-37) on a uniform grid dt = T / N, pseudo-random uniforms
// from ChaCha8Rng::seed_from_u64(seed_i + s) exactly as the generic kernel draws them.
//
// Scheduling: a persistent grid of waves pulls work items (instance, 64 * PPL paths) from an
// atomic counter. Items are queued longest-first (LPT on steps x paths), each wave reduces its
// item's terminal values to an f64 (sum, sum of squares) pair written to the item's fixed slot,
// and a finalize kernel reduces each instance's slots with Neumaier summation, so results do
// not depend on which wave ran which item. The counter is reset by a kernel (no memset), so the
// three launches can be captured into one hipGraph and replayed.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device/sdesim_device.hpp"
#include "reduce.hpp"

namespace {

// One Euler step of a built-in model. FP64 adds the terms to the state one at a time, in the
// reference's order (src/sim/euler.rs:20-27: the drift term, then the Wiener term), which keeps it
// bitwise equal to the DSL form's kernel.
template <bool LIB>
__device__ __forceinline__ double sde_euler_builtin(int kind, double x, double p0, double p1, double p2, double dt,
                                                    double sdt, double z) {
  double v0, v1;
  if (kind == 0) {
    v0 = p0 * x;
    v1 = p1 * x;
  } else if (kind == 1) {
    v0 = p0 * (p1 + (-x));
    v1 = p2;
  } else {
    v0 = p0 * (p1 + (-sde_fmax(x, 0.0)));
    if constexpr (LIB) v1 = p2 * sqrt(sde_fmax(x, 0.0));
    else v1 = p2 * sde_sqrt(sde_fmax(x, 0.0));
  }
  double a0 = x;
  a0 = a0 + v0 * dt;
  a0 = a0 + v1 * (sdt * z);
  return a0;
}
// FP32 sums the step's terms first and adds the sum to the state once, as the generated FP32 kernels do: added
// alone, a drift of a few ulps of x per step (GBM with mu dt ~ 3e-7) is rounded to whole ulps at every step in
// the same direction, which biased a 1000-step GBM mean by 1.5e-5. The products with dt and sqrt(dt) are
// the host's (f64, rounded once): GBM a = mu dt, b = sigma sqrt(dt); OU and CIR a = kappa dt, b = sigma
// sqrt(dt), and theta. 2, 4 and 8 operations instead of 6, 6 and 9.
template <int KIND>
__device__ __forceinline__ float sde_euler_builtin_f32(float x, float a, float b, float theta, float z) {
  if (KIND == 0) return x + x * (a + b * z);
  if (KIND == 1) return x + (a * (theta - x) + b * z);
  const float xp = sde_fmax(x, 0.0f);
  return x + (a * (theta - xp) + b * sde_sqrt(xp) * z);
}

// All steps of a wave's 64 * PPL paths in f64.
template <int PPL, bool LIB>
__device__ __forceinline__ void batch_steps(const sde_u32 (&key)[PPL][8], int N, int kind, double (&x)[PPL], double p0,
                                            double p1, double p2, double dt, double sdt) {
  for (int n0 = 0; n0 < N; n0 += 8) {
    sde_u32 blk[PPL][16];
#pragma unroll
    for (int j = 0; j < PPL; ++j) sde_chacha_block<8>(key[j], (sde_u64)(n0 / 8), blk[j]);
    // The draws are taken one by one (100 registers; all eight at once take 138).
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (n0 + i < N) {
#pragma unroll
        for (int j = 0; j < PPL; ++j) {
          const sde_u32 lo = blk[j][2 * i], hi = blk[j][2 * i + 1];
          double z;
          if constexpr (LIB) z = sde_inv_normal(sde_u01_from_words(lo, hi));
          else z = sde_psi_word(lo, hi);
          x[j] = sde_euler_builtin<LIB>(kind, x[j], p0, p1, p2, dt, sdt, z);
        }
      }
    }
  }
}

// All steps of a wave's 64 * PPL paths in f32: a loop per model, and whole ChaCha blocks' eight steps without
// a test between them.
template <int KIND, int PPL>
__device__ __forceinline__ void batch_steps_f32(const sde_u32 (&key)[PPL][8], int N, float (&x)[PPL], float a, float b,
                                                float theta) {
  for (int n0 = 0; n0 < N; n0 += 8) {
    float z[PPL][8];
#pragma unroll
    for (int j = 0; j < PPL; ++j) {
      sde_u32 blk[16], lo[8], hi[8];
      sde_chacha_block<8>(key[j], (sde_u64)(n0 / 8), blk);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        lo[i] = blk[2 * i];
        hi[i] = blk[2 * i + 1];
      }
      sde_psi_words<8>(lo, hi, z[j]);
    }
    if (n0 + 8 <= N) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
#pragma unroll
        for (int j = 0; j < PPL; ++j) x[j] = sde_euler_builtin_f32<KIND>(x[j], a, b, theta, z[j][i]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 7; ++i) {
        if (n0 + i < N) {
#pragma unroll
          for (int j = 0; j < PPL; ++j) x[j] = sde_euler_builtin_f32<KIND>(x[j], a, b, theta, z[j][i]);
        }
      }
    }
  }
}

template <typename R, int PPL>
__global__ void __launch_bounds__(256) sdesim_batch(const SdeInstance* __restrict__ inst,
                                                     const SdeItem* __restrict__ items, int n_items,
                                                     unsigned int* __restrict__ counter,
                                                     double* __restrict__ partials, R* __restrict__ terminal,
                                                     const long long* __restrict__ term_offset,
                                                     const void* __restrict__ normal_tab) {
  sde_normal_tab_load<R>(normal_tab);
  const int lane = threadIdx.x & 63;
  // A wave can never process more than n_items items, which bounds the loop whatever happens.
  for (int iter = 0; iter < n_items; ++iter) {
    // Claim the next item without a divergent branch: every lane adds (lane == 0) and lane 0's
    // result, the counter before this wave's claim, is made wave-uniform by readfirstlane (all
    // lanes are active at the loop head). The exit test is then a scalar branch of the whole wave.
    const unsigned int claim = atomicAdd(counter, lane == 0 ? 1u : 0u);
    const int k = (int)__builtin_amdgcn_readfirstlane(claim);
    if (k >= n_items) break;
    const SdeItem it = items[k];
    const SdeInstance I = inst[it.instance];
    const int N = I.steps;
    const int kind = I.kind;
    R x[PPL];
    sde_u32 key[PPL][8];
    long long sid[PPL];
    bool live[PPL];
#pragma unroll
    for (int j = 0; j < PPL; ++j) {
      const long long s = (long long)it.chunk * 64 * PPL + j * 64 + lane;
      live[j] = s < I.paths;
      sid[j] = live[j] ? s : 0;
      x[j] = (R)I.x0;
      sde_seed_from_u64(I.seed + (sde_u64)sid[j], key[j]);
    }
    if constexpr (sizeof(R) == 4) {
      if (kind == 0) batch_steps_f32<0, PPL>(key, N, x, I.af, I.bf, I.thetaf);
      else if (kind == 1) batch_steps_f32<1, PPL>(key, N, x, I.af, I.bf, I.thetaf);
      else batch_steps_f32<2, PPL>(key, N, x, I.af, I.bf, I.thetaf);
    } else if (kind == 2 && 4.0 * (I.p0 * I.p1) < I.p2 * I.p2) {
      // A CIR instance whose rounding differences grow (reaches_root in codegen.hpp) keeps the
      // library's logarithm, root and division.
      batch_steps<PPL, true>(key, N, kind, x, I.p0, I.p1, I.p2, I.dt, I.sdt);
    } else {
      batch_steps<PPL, false>(key, N, kind, x, I.p0, I.p1, I.p2, I.dt, I.sdt);
    }
    double acc[2] = {0.0, 0.0};
#pragma unroll
    for (int j = 0; j < PPL; ++j) {
      if (live[j]) {
        const double d = (double)x[j] - I.x0;
        acc[0] += d;
        acc[1] += d * d;
        if (terminal) terminal[term_offset[it.instance] + sid[j]] = x[j];
      }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) acc[i] += __shfl_xor(acc[i], off, 64);
    }
    if (lane == 0) {
      partials[2 * (long long)it.slot] = acc[0];
      partials[2 * (long long)it.slot + 1] = acc[1];
    }
  }
}

__global__ void sdesim_batch_reset(unsigned int* counter) {
  if (threadIdx.x == 0 && blockIdx.x == 0) counter[0] = 0u;
}

// G lanes per instance, whose item slots are [slot0[i], slot0[i+1]): a wave, or a thread where no instance has more than
// a few. (A wave each whatever the slots took 140 us more of 300,000 instances of one slot than a thread each; a
// thread each took 222 us of 4.2 ms where 4096 instances have hundreds.) Any number of blocks.
template <int G>
__global__ void __launch_bounds__(256) sdesim_batch_finalize(const SdeInstance* __restrict__ inst,
                                                             const int* __restrict__ slot0, int n,
                                                             const double* __restrict__ partials,
                                                             double* __restrict__ out) {
  const long long stride = (long long)gridDim.x * blockDim.x / G;
  const int lane = threadIdx.x & (G - 1);
  typedef double D2 __attribute__((ext_vector_type(2)));
  for (long long i = ((long long)blockIdx.x * blockDim.x + threadIdx.x) / G; i < n; i += stride) {
    SdeSum a, b;
    const int end = slot0[i + 1];
#pragma unroll 4
    for (int s = slot0[i] + lane; s < end; s += G) {
      const D2 v = *(const D2*)(partials + 2 * (long long)s);
      a.add(v.x);
      b.add(v.y);
    }
    if constexpr (G == 64) {
      sde_wave_sum(a);
      sde_wave_sum(b);
    }
    if (lane == 0) {
      const double S = (double)inst[i].paths;
      const double s1 = a.value(), s2 = b.value();
      const double m1 = s1 / S;
      out[2 * i] = inst[i].x0 + m1;
      out[2 * i + 1] = S > 1.0 ? (s2 - s1 * m1) / (S - 1.0) : 0.0;
    }
  }
}

}  // namespace

// Host launchers (batch runtime in runtime_batch.cpp).
hipError_t sdesim_launch_batch(int f32, int ppl, int grid, int block, const SdeInstance* inst, const SdeItem* items,
                               int n_items, unsigned int* counter, double* partials, void* terminal,
                               const long long* term_offset, const void* normal_tab, hipStream_t stream) {
  hipLaunchKernelGGL(sdesim_batch_reset, dim3(1), dim3(64), 0, stream, counter);
#define SDE_BATCH_CASE(R, P)                                                                            \
  if (ppl == P) {                                                                                        \
    hipLaunchKernelGGL((sdesim_batch<R, P>), dim3(grid), dim3(block), 0, stream, inst, items, n_items,     \
                       counter, partials, (R*)terminal, term_offset, normal_tab);                                \
    return hipGetLastError();                                                                            \
  }
  if (f32) {
    SDE_BATCH_CASE(float, 1)
    SDE_BATCH_CASE(float, 2)
    SDE_BATCH_CASE(float, 4)
  } else {
    SDE_BATCH_CASE(double, 1)
    SDE_BATCH_CASE(double, 2)
    SDE_BATCH_CASE(double, 4)
  }
#undef SDE_BATCH_CASE
  return hipErrorInvalidValue;
}

// most_slots: the largest number of slots of an instance. Up to 8, two rounds of a thread's loads in flight.
hipError_t sdesim_launch_batch_finalize(const SdeInstance* inst, const int* slot0, int n, int most_slots,
                                        const double* partials, double* out, hipStream_t stream) {
  const long long threads = most_slots <= 8 ? n : 64LL * n;
  const int grid = (int)std::min<long long>((threads + 255) / 256, 1 << 20);
  if (most_slots <= 8)
    hipLaunchKernelGGL(sdesim_batch_finalize<1>, dim3(grid), dim3(256), 0, stream, inst, slot0, n, partials, out);
  else
    hipLaunchKernelGGL(sdesim_batch_finalize<64>, dim3(grid), dim3(256), 0, stream, inst, slot0, n, partials, out);
  return hipGetLastError();
}

// Resident blocks per CU for a (precision, PPL, block) variant: sizes the persistent grid.
hipError_t sdesim_batch_occupancy(int f32, int ppl, int block, int* blocks_per_cu) {
#define SDE_OCC_CASE(R, P)                                                                                   \
  if (ppl == P) return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, sdesim_batch<R, P>, block, 0);
  if (f32) {
    SDE_OCC_CASE(float, 1)
    SDE_OCC_CASE(float, 2)
    SDE_OCC_CASE(float, 4)
  } else {
    SDE_OCC_CASE(double, 1)
    SDE_OCC_CASE(double, 2)
    SDE_OCC_CASE(double, 4)
  }
#undef SDE_OCC_CASE
  return hipErrorInvalidValue;
}
