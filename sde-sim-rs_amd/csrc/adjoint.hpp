// adjoint.hpp -- the state tape of the forward-rate model's reverse sweep; a reciprocal and a chunked
// per-block reduction of per-path results, shared with the basket.
//
// Tape layout [slot][row][path]: row r of a slot holds one state variable of every path. The ROWS rows
// of a slot sit under one buffer resource of ROWS * S * sizeof(R) bytes (below 2^31, checked by
// the host); the path's byte offset is the vector offset and the row's the scalar offset. Lanes
// past the last path pass vector offset 2^31, beyond the resource: their stores are dropped and
// their loads return 0, so no exec-masked branch surrounds the accesses. Both directions use the
// non-temporal policy: each value is written once and read once.
#pragma once

#include "device/sdesim_device.hpp"

// 1 / x: v_rcp_f32 (1 ulp), or the hardware seed (2^-24) and a third-order step (rounding of the
// last sum only; x is a growth or discount factor, far from f64's ends).
__device__ __forceinline__ float sde_recip(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ double sde_recip(double x) {
  const double y = __builtin_amdgcn_rcp(x), e = __builtin_fma(-x, y, 1.0);
  return __builtin_fma(y, __builtin_fma(e, e, e), y);
}

// One slot: its resource and a row's bytes. The latter is opaque to the compiler, which otherwise forms the
// ROWS row offsets once for the kernel, has no scalar registers for them and reads each from a vector
// register's lane at its use.
struct SdeTapeSlot {
  __amdgpu_buffer_rsrc_t rs;
  int row_bytes;
};

// n is wave-uniform; readfirstlane keeps the resource in scalar registers even where the index
// was formed by a vector instruction (a clamped subtraction, say), which would otherwise make
// the compiler wrap every access in a loop over distinct resources.
template <typename R, int ROWS>
__device__ __forceinline__ SdeTapeSlot sde_tape_slot(void* tape, int n, long long S) {
  n = __builtin_amdgcn_readfirstlane(n);
  const long long slot_bytes = (long long)ROWS * S * (long long)sizeof(R);
  SdeTapeSlot t;
  t.rs = __builtin_amdgcn_make_buffer_rsrc((void*)((char*)tape + (long long)n * slot_bytes), (short)0, (int)slot_bytes,
                                           0x00020000);
  t.row_bytes = (int)(S * (long long)sizeof(R));
  asm volatile("" : "+s"(t.row_bytes));
  return t;
}

template <typename R>
__device__ __forceinline__ R sde_tape_get(const SdeTapeSlot& t, sde_u32 voff, int row) {
  if constexpr (sizeof(R) == 4)
    return __builtin_bit_cast(float, (sde_u32)__builtin_amdgcn_raw_buffer_load_b32(t.rs, (int)voff, row * t.row_bytes, 2));
  else
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(t.rs, (int)voff, row * t.row_bytes, 2));
}

// Row `row` of a slot, with cache policy AUX.
template <typename R, int AUX>
__device__ __forceinline__ void sde_tape_put(const SdeTapeSlot& t, sde_u32 voff, int row, R x) {
  if constexpr (sizeof(R) == 4)
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(sde_u32, (float)x), t.rs, (int)voff, row * t.row_bytes, AUX);
  else
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(SdeU32x2, (double)x), t.rs, (int)voff, row * t.row_bytes, AUX);
}

template <typename R, int ROWS>
__device__ __forceinline__ void sde_tape_store(void* tape, int n, long long S, sde_u32 voff, const R (&X)[ROWS]) {
  const SdeTapeSlot t = sde_tape_slot<R, ROWS>(tape, n, S);
#pragma unroll
  for (int i = 0; i < ROWS; ++i) sde_tape_put<R, 2>(t, voff, i, X[i]);
}

template <typename R, int ROWS>
__device__ __forceinline__ void sde_tape_load(void* tape, int n, long long S, sde_u32 voff, R (&X)[ROWS]) {
  const SdeTapeSlot t = sde_tape_slot<R, ROWS>(tape, n, S);
#pragma unroll
  for (int i = 0; i < ROWS; ++i) X[i] = sde_tape_get<R>(t, voff, i);
}

// One partial per block of each of the NQ per-path values get(q): a butterfly over the wave's
// lanes, then the waves in order (the summation order of sde_block_reduce_store), eight
// quantities at a time so that only eight f64 values per lane are live.
template <int NQ, class G>
__device__ __forceinline__ void sde_reduce_store_chunked(const G& get, double* __restrict__ out) {
  __shared__ double red[16][8];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int nw = (blockDim.x + 63) >> 6;
#pragma unroll
  for (int q0 = 0; q0 < NQ; q0 += 8) {
    double v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = q0 + i < NQ ? get(q0 + i) : 0.0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) v[i] += __shfl_xor(v[i], off, 64);
    }
    if (lane == 0) {
#pragma unroll
      for (int i = 0; i < 8; ++i) red[wave][i] = v[i];
    }
    __syncthreads();
    if ((int)threadIdx.x < 8 && q0 + (int)threadIdx.x < NQ) {
      double t = 0.0;
      for (int w = 0; w < nw; ++w) t += red[w][threadIdx.x];
      out[q0 + threadIdx.x] = t;
    }
    __syncthreads();
  }
}
