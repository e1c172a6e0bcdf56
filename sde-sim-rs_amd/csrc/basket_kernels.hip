// basket_kernels.hip -- correlated GBM basket: price and pathwise derivatives, summed on the way forward.
//
// Model: A assets, X_{n+1,i} = X_{n,i} + X_{n,i} (mu_i dt + sigma_i sqrt(dt) Z_{n,i}),
// Z_n = L eps_n with L the lower Cholesky factor of the correlation and eps_{n,k} = Psi(u_{n,k})
// (A&S inverse normal, src/proc/increment.rs:160-179) of the pseudo-random draw n*A + k of
// ChaCha8Rng::seed_from_u64(seed + s) -- the Euler step of the reference (src/sim/euler.rs:5-37)
// applied to the DSL form dX_i = (mu_i * X_i) * dt + sum_k (sigma_i * L_ik * X_i) * dW_k.
// Payoff on the weighted basket B = sum_i w_i X_{N,i}: width * softplus((B - K) / width), or the
// plain call max(B - K, 0) when width == 0.
//
// Adjoint (no reference counterpart): pathwise derivatives of the payoff with respect to X0, mu,
// sigma and L, per path, reduced over paths in f64, all accumulated on the way forward. With
//   g_{n,i} = X_{n+1,i} / X_{n,i} = 1 + mu_i dt + sigma_i sqrt(dt) Z_{n,i}
// the reverse recursion Xbar_n = Xbar_{n+1} g_n makes M_i = Xbar_{n,i} X_{n,i} the same for every n, so it is
// known from the final state (payoff' w_i X_{N,i}), and what a step adds to a derivative is M_i times a
// quantity of that step alone:
//   X0bar_i = M_i / X0_i,  mubar_i = M_i dt sum_n 1 / g_{n,i},
//   Lbar_ik = M_i sigma_i sqrt(dt) H_ik,  H_ik = sum_n eps_{n,k} / g_{n,i}  (k <= i),
//   sigmabar_i = M_i sqrt(dt) sum_{k <= i} L_ik H_ik.
// A growth of exactly 0 (mu_i dt + sigma_i sqrt(dt) Z rounding to -1, once in 1e8 draws of a coarse f32
// grid) leaves M_i = 0 and 1 / g infinite, where the derivatives are finite. The block's partials are then NaN,
// which the host sees in the sums, and sdesim_basket_again takes such blocks again in the form that keeps
// the zero out of the product (step_careful): no test of a growth in the loop of every other run.
// No state is kept. The reverse sweep that this replaces wrote and read every state (49 GB for 8 assets x
// 365 steps x 2^22 paths in f32): 26.1 ms for price and Greeks, 17.6 ms now, bound by VALU issue: a step's 8
// draws are two thirds of it (350 instructions of ChaCha8, 80 of the normals), the 36 sums, 8
// reciprocals and the step the rest.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "device/sdesim_device.hpp"
#include "adjoint.hpp"
#include "reduce.hpp"

namespace {

template <int D>
struct BasketConst {
  static constexpr int NL = D * (D + 1) / 2;   // lower-triangular entries of L
  static constexpr int NQ = 2 + 3 * D + NL;    // reduced quantities: payoff, payoff^2, gradients
};

// f(0), f(1), .. f(N - 1) with the argument a constant.
template <int I, int N, class F>
__device__ __forceinline__ void basket_static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    basket_static_for<I + 1, N>(f);
  }
}

// The path's normals in order, taken with compile-time positions: draw(j) for j = 0, 1, .. of a chunk
// of steps that starts on a block. f32 converts a block's eight draws together (one test for rare
// ones), f64 each on its own (fewer registers).
template <typename R>
struct BasketNormals {
  sde_u32 lo[8], hi[8];
  float z[8];
  template <int j>
  __device__ __forceinline__ R draw(const sde_u32 (&key)[8], sde_u64 block0) {
    if constexpr (j % 8 == 0) {
      sde_u32 blk[16];
      sde_chacha_block<8>(key, block0 + (sde_u64)(j / 8), blk);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        lo[k] = blk[2 * k];
        hi[k] = blk[2 * k + 1];
      }
      if constexpr (sizeof(R) == 4) sde_psi_words<8>(lo, hi, z);
    }
    if constexpr (sizeof(R) == 4) return z[j % 8];
    else return sde_psi_word(lo[j % 8], hi[j % 8]);
  }
};

template <typename R>
__device__ __forceinline__ R basket_softplus(R x) {
  // log(1 + e^x) without overflow: max(x, 0) + log1p(exp(-|x|))
  return (x > R(0) ? x : R(0)) + (R)log1p(exp(-(double)fabs((double)x)));
}

// Payoff of the weighted basket at the final state and its derivative with respect to B.
template <typename R, int D>
__device__ __forceinline__ void basket_payoff(const R (&X)[D], const R (&w)[D], R K, R width, R& pay, R& dpay) {
  R B = R(0);
#pragma unroll
  for (int i = 0; i < D; ++i) B = B + w[i] * X[i];
  if (width > R(0)) {
    const R x = (B - K) / width;
    pay = width * basket_softplus<R>(x);
    dpay = (R)(1.0 / (1.0 + exp(-(double)x)));
  } else {
    pay = B > K ? B - K : R(0);
    dpay = B > K ? R(1) : R(0);
  }
}

// The step's parameters in the path precision, in scalar registers: mu dt and sigma sqrt(dt) L.
template <typename R>
__device__ __forceinline__ R basket_mdt(const BasketArgs& a, int i) {
  if constexpr (sizeof(R) == 4) return a.mdt_f[i];
  else return a.mdt[i];
}
template <typename R>
__device__ __forceinline__ R basket_scl(const BasketArgs& a, int i, int k) {
  if constexpr (sizeof(R) == 4) return a.scl_f[i * 8 + k];
  else return a.scl[i * 8 + k];
}

// A path: the state, the sums H of the header and sum_n 1 / g_n.
template <typename R, int D, bool ADJ>
struct BasketPath {
  static constexpr int NL = BasketConst<D>::NL, NQ = BasketConst<D>::NQ;
  R X[D], H[NL], Q[D];

  __device__ __forceinline__ explicit BasketPath(const BasketArgs& a) {
#pragma unroll
    for (int i = 0; i < D; ++i) {
      X[i] = (R)a.x0[i];
      Q[i] = R(0);
    }
#pragma unroll
    for (int q = 0; q < NL; ++q) H[q] = R(0);
  }

  __device__ __forceinline__ void step(const BasketArgs& a, const R (&eps)[D]) {
#pragma unroll
    for (int i = 0; i < D; ++i) {
      R c = basket_mdt<R>(a, i);
#pragma unroll
      for (int k = 0; k <= i; ++k) c = c + basket_scl<R>(a, i, k) * eps[k];
      X[i] = X[i] + X[i] * c;
      if constexpr (ADJ) {
        const R r = sde_recip(R(1) + c);
        Q[i] = Q[i] + r;
#pragma unroll
        for (int k = 0; k <= i; ++k) H[i * (i + 1) / 2 + k] = H[i * (i + 1) / 2 + k] + r * eps[k];
      }
    }
  }

  // The same step where growths may be 0. With one zero in the product only the zero's own step has a derivative, M_i
  // there being the product of the other growths, so the sums start anew from that step and are closed by it; a
  // second zero makes M_i 0.
  __device__ __forceinline__ void step_careful(const BasketArgs& a, const R (&eps)[D], sde_u32& zeroed) {
#pragma unroll
    for (int i = 0; i < D; ++i) {
      R c = basket_mdt<R>(a, i);
#pragma unroll
      for (int k = 0; k <= i; ++k) c = c + basket_scl<R>(a, i, k) * eps[k];
      const bool zero = R(1) + c == R(0), past = ((zeroed >> i) & 1u) != 0u;
      const R keep = zero && !past ? R(0) : R(1), r = past ? R(0) : zero ? R(1) : sde_recip(R(1) + c);
      X[i] = X[i] + X[i] * (!zero ? c : past ? R(-1) : R(0));
      Q[i] = Q[i] * keep + r;
#pragma unroll
      for (int k = 0; k <= i; ++k) H[i * (i + 1) / 2 + k] = H[i * (i + 1) / 2 + k] * keep + r * eps[k];
      zeroed |= zero ? 1u << i : 0u;
    }
  }

  // The block's partials: price (payoff and payoff^2) or, with ADJ, price and derivatives, of the paths whose
  // lanes have `live` set. All threads take part. ZEROED: bit i of `zeroed` is set when a growth of asset i was 0, and
  // X[i] is the product of the others.
  template <bool ZEROED = false>
  __device__ __forceinline__ void finish(const BasketArgs& a, bool live, sde_u32 zeroed = 0u) {
    R w[D];
#pragma unroll
    for (int i = 0; i < D; ++i) w[i] = (R)a.weight[i];
    R pay, dpay;
    if constexpr (ZEROED) {
      R XN[D];
#pragma unroll
      for (int i = 0; i < D; ++i) XN[i] = (zeroed >> i) & 1u ? R(0) : X[i];
      basket_payoff<R, D>(XN, w, (R)a.strike, (R)a.width, pay, dpay);
    } else {
      basket_payoff<R, D>(X, w, (R)a.strike, (R)a.width, pay, dpay);
    }
    if constexpr (ADJ) {
      R m[D], lh[D];
#pragma unroll
      for (int i = 0; i < D; ++i) {
        m[i] = dpay * w[i] * X[i];
        lh[i] = R(0);
#pragma unroll
        for (int k = 0; k <= i; ++k) lh[i] = lh[i] + (R)a.chol[i * 8 + k] * H[i * (i + 1) / 2 + k];
      }
      const R dt = (R)a.dt, sdt = (R)a.sdt;
      // Derivative q of this path, q < 3 D + NL: d/dX0, d/dmu, d/dsigma, d/dL (q a constant after
      // unrolling).
      auto grad = [&](int q) -> double {
        if (ZEROED && q < D && ((zeroed >> q) & 1u)) return (double)(R(0) / (R)a.x0[q]);
        if (q < D) return (double)(m[q] / (R)a.x0[q]);
        if (q < 2 * D) return (double)(m[q - D] * dt * Q[q - D]);
        if (q < 3 * D) return (double)(m[q - 2 * D] * sdt * lh[q - 2 * D]);
        int i = 0;
        while ((i + 1) * (i + 2) / 2 <= q - 3 * D) ++i;
        return (double)(m[i] * ((R)a.sigma[i] * sdt) * H[q - 3 * D]);
      };
      sde_reduce_store_chunked<NQ>(
          [&](int q) { return !live ? 0.0 : q == 0 ? (double)pay : q == 1 ? (double)pay * (double)pay : grad(q - 2); },
          a.partials + (long long)blockIdx.x * NQ);
    } else {
      sde_reduce_store_chunked<2>(
          [&](int q) { return !live ? 0.0 : q == 0 ? (double)pay : (double)pay * (double)pay; },
          a.partials + (long long)blockIdx.x * 2);
    }
  }
};

// One path per lane. f32 is held to 4 waves per SIMD (128 VGPRs): 8 assets with Greeks take 139 unconstrained;
// with 11 values spilled (a load or store of each a step) they take 17.63 instead of 17.95 ms.
template <typename R, int D, bool ADJ>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sizeof(R) == 4 ? 4 : 1)))
sdesim_basket(const BasketArgs a) {
  constexpr int U = SdeChunk<D>::U;  // steps in a whole number of ChaCha blocks
  sde_normal_tab_load<R>(a.normal_tab);
  const int N = a.steps;
  const long long s = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = s < a.paths;

  sde_u32 key[8];
  sde_seed_from_u64(a.seed + (sde_u64)(live ? s : 0), key);
  BasketPath<R, D, ADJ> path(a);
  for (int n0 = 0; n0 < N; n0 += U) {
    BasketNormals<R> noise;
    basket_static_for<0, U>([&](auto u_) {
      constexpr int u = u_;
      if (U == 1 || n0 + u < N) {
        R eps[D];
        basket_static_for<0, D>([&](auto k_) {
          constexpr int k = k_;
          eps[k] = noise.template draw<u * D + k>(key, (sde_u64)n0 * D / 8);
        });
        path.step(a, eps);
      }
    });
  }
  path.finish(a, live);
}

// Few paths: a block of four waves, one per SIMD of a CU, for 64 of them, as sde_team_kernel has it. Waves 0
// to 2 put the normals of a round's ChaCha blocks into LDS, the last wave steps the paths through those of
// the round before. A round is about six blocks of a whole number of steps. With Greeks: 7 assets in f32, 10,000
// paths x 365 steps, 0.25 instead of 0.46 ms for the call; 5 in f64, 30,001 x 252, 0.32 instead of 0.38.
template <typename R, int D, bool ADJ>
__global__ void __launch_bounds__(256) sdesim_basket_team(const BasketArgs a) {
  constexpr int U = SdeChunk<D>::U, NB = SdeChunk<D>::BLOCKS;
  constexpr int UNITS = NB == 1 ? 6 : NB == 3 ? 2 : 1;  // of U steps (NB blocks) in a round
  __shared__ R noise[2][UNITS * NB * 8][64];
  sde_normal_tab_load<R>(a.normal_tab);
  const int N = a.steps;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const long long s = (long long)blockIdx.x * 64 + lane;
  const bool live = s < a.paths, steps = wave == 3;

  sde_u32 key[8];
  sde_seed_from_u64(a.seed + (sde_u64)(live ? s : 0), key);
  BasketPath<R, D, ADJ> path(a);
  if (steps) __builtin_amdgcn_s_setprio(3);  // it shares its SIMD with other blocks' producers
  // Every wave passes every barrier: the trip count is the same for all.
  const int rounds = (N + UNITS * U - 1) / (UNITS * U);
  for (int r = 0; r <= rounds; ++r) {
    if (!steps) {
      for (int b = wave; b < UNITS * NB; b += 3) {
        const long long block = (long long)r * (UNITS * NB) + b;
        if (r < rounds && block * 8 < (long long)N * D) {
          sde_u32 blk[16], lo[8], hi[8];
          R z[8];
          sde_chacha_block<8>(key, (sde_u64)block, blk);
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            lo[k] = blk[2 * k];
            hi[k] = blk[2 * k + 1];
          }
          sde_psi_words<8>(lo, hi, z);
#pragma unroll
          for (int k = 0; k < 8; ++k) noise[r & 1][b * 8 + k][lane] = z[k];
        }
      }
    } else if (r > 0) {
      for (int q = 0; q < UNITS; ++q) {
        const int n0 = ((r - 1) * UNITS + q) * U;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (n0 + u < N) {
            R eps[D];
#pragma unroll
            for (int k = 0; k < D; ++k) eps[k] = noise[(r - 1) & 1][(q * U + u) * D + k][lane];
            path.step(a, eps);
          }
        }
      }
    }
    __syncthreads();
  }
  path.finish(a, steps && live);
}

// The blocks whose partials of the derivatives are not all finite, once more: same paths, step_careful. blockDim is the
// first kernel's paths a block.
template <typename R, int D>
__global__ void __launch_bounds__(256) sdesim_basket_again(const BasketArgs a) {
  constexpr int NQ = BasketConst<D>::NQ, U = SdeChunk<D>::U;
  const int N = a.steps;
  bool finite = true;
  for (int q = 2; q < NQ; ++q) {
    const double v = a.partials[(long long)blockIdx.x * NQ + q];
    finite = finite && v - v == 0.0;
  }
  if (finite) return;  // the whole block
  __syncthreads();     // every wave has read the partials that finish() replaces
  sde_normal_tab_load<R>(a.normal_tab);
  const long long s = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = s < a.paths;
  sde_u32 key[8];
  sde_seed_from_u64(a.seed + (sde_u64)(live ? s : 0), key);
  BasketPath<R, D, true> path(a);
  sde_u32 zeroed = 0u;
  for (int n0 = 0; n0 < N; n0 += U) {
    BasketNormals<R> noise;
    basket_static_for<0, U>([&](auto u_) {
      constexpr int u = u_;
      if (U == 1 || n0 + u < N) {
        R eps[D];
        basket_static_for<0, D>([&](auto k_) {
          constexpr int k = k_;
          eps[k] = noise.template draw<u * D + k>(key, (sde_u64)n0 * D / 8);
        });
        path.step_careful(a, eps, zeroed);
      }
    });
  }
  path.template finish<true>(a, live, zeroed);
}

// Sum of per-block partials per quantity: one block of 1024 threads each, whose loads of 8 bytes
// from rows of nq values are all in flight together (the quantities' blocks read the same lines
// through L2).
__global__ void __launch_bounds__(1024) sdesim_sum_partials(const double* __restrict__ partials, int nblocks, int nq,
                                                            double* __restrict__ out) {
  const int q = blockIdx.x;
  SdeSum a;
#pragma unroll 8
  for (int b = threadIdx.x; b < nblocks; b += blockDim.x) a.add(partials[(long long)b * nq + q]);
  __shared__ double sh[16][2];
  sde_block_sum(a, sh);
  if (threadIdx.x == 0) out[q] = a.value();
}

}  // namespace

hipError_t sdesim_launch_sum_partials(const double* partials, int nblocks, int nq, double* out, hipStream_t stream) {
  hipLaunchKernelGGL(sdesim_sum_partials, dim3(nq), dim3(nblocks > 256 ? 1024 : 256), 0, stream, partials, nblocks, nq, out);
  return hipGetLastError();
}

// team: 64 paths a block (sdesim_basket_team), else 256. again: the blocks whose partials are not finite (after an
// adjoint run). A kernel per asset count, which draws, correlates and sums no more than the basket's own assets: padded to 8
// assets, 5 in f64 took three times as long.
hipError_t sdesim_launch_basket(int f32, int assets, int adjoint, int team, int again, int grid, const BasketArgs& a,
                                int nq, double* sums, hipStream_t stream) {
#define SDE_BASKET(R, D, ADJ)                                                                                     \
  do {                                                                                                            \
    if (again) hipLaunchKernelGGL((sdesim_basket_again<R, D>), dim3(grid), dim3(team ? 64 : 256), 0, stream, a);  \
    else if (team) hipLaunchKernelGGL((sdesim_basket_team<R, D, ADJ>), dim3(grid), dim3(256), 0, stream, a);           \
    else hipLaunchKernelGGL((sdesim_basket<R, D, ADJ>), dim3(grid), dim3(256), 0, stream, a);                     \
  } while (0)
#define SDE_BASKET_WIDTH(D)                         \
  case D:                                           \
    if (f32 && adjoint) SDE_BASKET(float, D, true); \
    else if (f32) SDE_BASKET(float, D, false);      \
    else if (adjoint) SDE_BASKET(double, D, true);  \
    else SDE_BASKET(double, D, false);              \
    break;
  switch (assets) {
    SDE_BASKET_WIDTH(1)
    SDE_BASKET_WIDTH(2)
    SDE_BASKET_WIDTH(3)
    SDE_BASKET_WIDTH(4)
    SDE_BASKET_WIDTH(5)
    SDE_BASKET_WIDTH(6)
    SDE_BASKET_WIDTH(7)
    SDE_BASKET_WIDTH(8)
    default: return hipErrorInvalidValue;
  }
#undef SDE_BASKET_WIDTH
#undef SDE_BASKET
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return sdesim_launch_sum_partials(a.partials, grid, nq, sums, stream);
}
