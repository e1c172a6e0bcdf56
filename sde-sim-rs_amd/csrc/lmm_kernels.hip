// lmm_kernels.hip -- multi-factor forward-rate (LIBOR market) model: swaption price and pathwise
// curve sensitivities. No reference counterpart (the reference has no built-in models and no
// sensitivities); the stepping is log-Euler with uniforms from the same scrambled Sobol stream
// as the generic kernel (src/rng/sobol.rs points, XOR digital shift) and the A&S inverse normal
// (src/proc/increment.rs:160-179).
//
// Forwards L_i on [T_i, T_{i+1}], T_i = i * tau, i = 0 .. NF-1, NF = 40; F = 3 factors with
// loadings B (NF x F, unit rows); volatilities sig_i. Spot measure: at step n (t_n = n dt) the
// alive forwards are i >= eta = n / steps_per_period + 1, and for them
//   ln L_i += (sig_i sum_f B_if C_f(i) - sig_i^2 / 2) dt + sig_i sqrt(dt) sum_f B_if eps_f,
//   C_f(i) = sum_{j=eta..i} tau sig_j L_j / (1 + tau L_j) B_jf     (a prefix sum over j),
// eps_f = Psi(u_{n F + f}). Dead forwards keep their fixing value.
// Payoff at expiry T_e (e = expiry index): receiver swaption on the swap over [T_e, T_NF] with
// fixed rate K: V = max(K A - (1 - P_{NF-1}), 0) / N, P_j = prod_{k=e..j} 1 / (1 + tau L_k),
// A = tau sum_{j=e..NF-1} P_j, numeraire N = prod_{k<e} (1 + tau L_k).
//
// What a forward is held by, H_i: its growth P_i = L_i / L_i(0) in f32, tau L_i in f64. The f32 state is y_i = log2
// P_i: a step adds to it, and what rounds at every step is a sum below 1. Multiplying P_i by the step's exponential
// costs as much, and v_exp_f32's mean error (-1e-9 to -4e-9 next to 1) adds up over the steps: the f32 price was
// 6.1e-7 off over 160 steps and 2.1e-7 over 40, always to one side; now 2.5e-8 and 1e-8. In f64 the state is H_i itself,
// which the drift needs no parameter to use: with growths, the wait for the parameter row came before the
// reciprocal (price 3 % slower).
//
// Adjoint: with M_i = dV/dH_i H_i / c_i, c_i = L_i(0) in f32 (M_i is then the derivative with respect to L_i(0) as far
// as it goes through forward i's own factor) and 1 in f64 (the host divides the sums by L_i(0)), one step back is,
// H the state before it,
//   G_f(j) = sum_{i >= j} M'_i c_i sig_i B_if (a suffix sum),
//   M_j = M'_j + dt (sum_f B_jf G_f(j)) tau sig_j L_j / c_j / (1 + tau L_j)^2,
// which needs neither the state after the step nor a quotient of the two. The states come from
//  * the state tape (MODE 2): the forward pass writes every second H, H_0, H_2, .. and H_N, to HBM
//    ([slot][i][path], 13.6 GB for 160 steps x 40 forwards x 2^20 paths in f32; forwards that are dead by then
//    only in H_N); a second kernel reads them back and recomputes the states between;
//  * checkpoints (MODE 1): the forward pass stores the state every SEG steps ([slot][i][path]); the
//    reverse sweep takes the segments last to first, recomputes a segment's H once from its
//    checkpoint into the segment tape ([k][i][path], rewritten per segment) and then steps back
//    through them.
// Price and sensitivities at that size, f32: 6.75 ms a call, VALU issue and the chains within a step; 9.7 with every state
// on the tape and a step back that holds the states on both sides of it: both kernels then waited for HBM. The
// price alone: 2.57 (2.51 as products of exponentials).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "device/sdesim_device.hpp"
#include "adjoint.hpp"

namespace {

constexpr int NF = 40;
constexpr int F = 3;
constexpr int SEG = 16;  // checkpoint interval (~sqrt of the 160-step workload)
constexpr float LMM_ROOT_LOG2E = SDE_LMM_ROOT_LOG2E;  // s of the parameter rows
constexpr int NSL = 3;  // Sobol table slices: point indices below 2^22

// exp of an exponent given in the parameter rows' units: base 2 for f32 (the rows carry the
// log2(e) factor, so this is one v_exp_f32), natural for f64.
template <typename R>
__device__ __forceinline__ R lmm_exp_row(R x) {
  if constexpr (sizeof(R) == 4) return __builtin_amdgcn_exp2f(x);
  else return exp(x);
}

// H of a state, and the state after a step of exponent x.
template <typename R>
__device__ __forceinline__ R lmm_held(R y) {
  if constexpr (sizeof(R) == 4) return lmm_exp_row<R>(y);
  else return y;
}
template <typename R>
__device__ __forceinline__ R lmm_advance(R y, R x) {
  if constexpr (sizeof(R) == 4) return y + x;
  else return y * lmm_exp_row<R>(x);
}

// Where a lane's Sobol words live: its slice-0 entry (byte offset within a step's [64][F] block)
// and the wave's rows of slices 1-2 (the wave's 64 point indices share those Gray-code bits).
struct LmmSobol {
  sde_u32 voff0;
  sde_const_u32* urow[NSL - 1];
};

// The F uniforms of step n (digital XOR shift folded into the tables: the XOR of the slices is the
// complement of the scrambled point), as standard normals times s (LmmRow): one vector load of the lane's F
// slice-0 words and scalar loads of the wave's words of slices 1-2.
template <typename R>
__device__ __forceinline__ void lmm_noise(__amdgpu_buffer_rsrc_t rsrc, const LmmSobol& sb, int n, R (&eps)[F]) {
  sde_u32 w[F];
  sde_load_words<F>(rsrc, (int)sb.voff0, n * (64 * F * 4), w);
#pragma unroll
  for (int f = 0; f < F; ++f) {
    SdeUnifX u;
    u.yc = w[f] ^ sb.urow[0][n * F + f] ^ sb.urow[1][n * F + f];
    u.tail = nullptr;
    u.sm = u.sm2 = 0x80000000u;
    eps[f] = sde_psi<R>(u);
    if constexpr (sizeof(R) == 4) eps[f] = eps[f] * LMM_ROOT_LOG2E;
  }
}

// Model parameters: one 8-value row per forward with the step's constant products precomputed, in device
// memory, read with scalar loads so that a row's values are scalar operands of the arithmetic. Each
// step reads them at a pointer the compiler cannot see through: the reads repeat per step (and hit the
// scalar cache) instead of 320 loop-invariant values being hoisted and spilled. From LDS, two
// broadcast reads per forward took as long as the forward's arithmetic (16 cycles of the CU's LDS for a
// wave, against 60 of one of its four SIMDs).
template <typename R>
using LmmRow = R __attribute__((ext_vector_type(8)));
//       forward rows                        step back
//   0   tau L_i(0) (f32 only)               tau L_i(0) (f32 only)
//   1   q = sigma_i B_if sqrt(dt) un / s    loadings B_if
//   4   h = -sigma_i^2 dt / 2 un            c_i sigma_i B_if
//   7                                       tau sigma_i dt in f32, sigma_i dt in f64
// un is 1, or log2 e for f32, whose exponential has base 2; s is its root, rounded to f32, by which the step's normals
// are multiplied, so that q serves the drift's sums and the exponent. (q is formed with the rounded s and
// rounded once itself: a rounding of s alone would be common to every forward and step.)
template <typename R>
using LmmRows = __attribute__((address_space(4))) const LmmRow<R>*;
typedef __attribute__((address_space(4))) const double* LmmDoubles;
template <typename T>
__device__ __forceinline__ T lmm_opaque(const void* at) {
  sde_u64 p = (sde_u64)at;
  asm volatile("" : "+s"(p));
  return (T)p;
}
template <typename R>
__device__ __forceinline__ LmmRows<R> lmm_rows(const void* rows) {
  return lmm_opaque<LmmRows<R>>(rows);
}

// f(i, rows, C) for runs of C alive forwards from i upwards, or from i + C - 1 downwards: C is 4 for a group of four
// with no dead forward, which has no branch inside, so the forwards' chains overlap, and loads its rows together;
// otherwise 1. The second test is on a copy of eta that the compiler does not know to be one: joined into an
// if and else, the two sides' results would meet in copies of all the state.
template <typename R, bool DOWN, class Fn>
__device__ __forceinline__ void lmm_alive(LmmRows<R> rows, int eta, const Fn& f) {
  int eta2 = eta;
  asm volatile("" : "+s"(eta2));
#pragma unroll
  for (int g = 0; g < NF / 4; ++g) {
    const int i0 = 4 * (DOWN ? NF / 4 - 1 - g : g);
    if (i0 >= eta) f(i0, rows + i0, std::integral_constant<int, 4>{});
    if (i0 < eta2 && i0 + 3 >= eta2) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = DOWN ? i0 + 3 - j : i0 + j;
        if (i >= eta2) f(i, rows + i, std::integral_constant<int, 1>{});
      }
    }
  }
}

// tau L_i from its parameter row and H_i.
template <typename R>
__device__ __forceinline__ R lmm_tau_L(const LmmRow<R>& r, R H) {
  if constexpr (sizeof(R) == 4) return r[0] * H;
  else return H;
}

// The exponents x of C forwards of which H is given. With D_f = s eps_f + sqrt(dt) C_f un / s, kept as one running
// sum over the forwards, the exponent is q_i.D + h_i. The C reciprocals come first: one after the other, as the
// compiler has it by itself, they are waited for.
template <typename R, int C>
__device__ __forceinline__ void lmm_exponents(LmmRows<R> rows, const R (&H)[C], R (&D)[F], R (&x)[C]) {
  R v[C];
#pragma unroll
  for (int j = 0; j < C; ++j) {
    const LmmRow<R> r = rows[j];
    const R w = lmm_tau_L<R>(r, H[j]);
    v[j] = w * sde_recip(R(1) + w);
  }
#pragma unroll
  for (int j = 0; j < C; ++j) {
    const LmmRow<R> r = rows[j];
#pragma unroll
    for (int f = 0; f < F; ++f) D[f] = D[f] + v[j] * r[1 + f];
    x[j] = r[1] * D[0] + r[2] * D[1] + r[3] * D[2] + r[4];
  }
}

// One log-Euler step of all alive forwards (those below `eta` are dead, and left alone); put(i, H_i) is given
// the H before it.
template <typename R, class Put>
__device__ __forceinline__ void lmm_step(LmmRows<R> rows, R (&Y)[NF], const R (&eps)[F], int eta, const Put& put) {
  R D[F] = {eps[0], eps[1], eps[2]};
  lmm_alive<R, false>(rows, eta, [&](int i, LmmRows<R> r, auto count) {
    constexpr int C = count;
    R H[C], x[C];
#pragma unroll
    for (int j = 0; j < C; ++j) {
      H[j] = lmm_held<R>(Y[i + j]);
      put(i + j, H[j]);
    }
    lmm_exponents<R, C>(r, H, D, x);
#pragma unroll
    for (int j = 0; j < C; ++j) Y[i + j] = lmm_advance<R>(Y[i + j], x[j]);
  });
}

// The same step from H to H.
template <typename R>
__device__ __forceinline__ void lmm_step_held(LmmRows<R> rows, const R (&H)[NF], R (&Hp)[NF], const R (&eps)[F], int eta) {
  R D[F] = {eps[0], eps[1], eps[2]};
  lmm_alive<R, false>(rows, eta, [&](int i, LmmRows<R> r, auto count) {
    constexpr int C = count;
    R h[C], x[C];
#pragma unroll
    for (int j = 0; j < C; ++j) h[j] = H[i + j];
    lmm_exponents<R, C>(r, h, D, x);
#pragma unroll
    for (int j = 0; j < C; ++j) Hp[i + j] = h[j] * lmm_exp_row<R>(x[j]);
  });
}

// One step back: H before the step; M on entry that of the state after it.
template <typename R>
__device__ __forceinline__ void lmm_step_back(LmmRows<R> rows, const R (&H)[NF], R (&M)[NF], int eta) {
  R G[F] = {R(0), R(0), R(0)};
  lmm_alive<R, true>(rows, eta, [&](int i0, LmmRows<R> rs, auto count) {
    constexpr int C = count;
#pragma unroll
    for (int j = C - 1; j >= 0; --j) {
      const int i = i0 + j;
      const LmmRow<R> r = rs[j];
#pragma unroll
      for (int f = 0; f < F; ++f) G[f] = G[f] + M[i] * r[4 + f];
      const R ab = r[1] * G[0] + r[2] * G[1] + r[3] * G[2];
      const R rop = sde_recip(R(1) + lmm_tau_L<R>(r, H[i]));
      M[i] = M[i] + ab * (r[7] * H[i] * rop * rop);
    }
  });
}

// Payoff at the final H (discounted by the spot numeraire) and, with GRAD, M_k: the numeraire part for k < e, the swap part for k >= e (only when in the money). In f64
// for f32 paths too: 36 rounded discount factors left the swap's value 3e-7 off, which decided on the wrong
// side for a path or two in 2^20, each 1e-6 of a sensitivity. It is one part in 100 of the path's work.
template <typename R, bool GRAD>
__device__ __forceinline__ double lmm_payoff(const LmmArgs& a, const R (&H)[NF], R (&M)[NF]) {
  const int e = a.expiry_index;
  const double tau = a.tau, K = a.strike;
  const LmmDoubles tau_L0 = lmm_opaque<LmmDoubles>(a.tau_L0);  // read here, not held in 80 registers from the start
  auto tau_L = [&](int k) -> double {
    if constexpr (sizeof(R) == 4) return tau_L0[k] * (double)H[k];
    else return H[k];
  };
  double numer = 1.0, Q = 1.0, A = 0.0;
#pragma unroll
  for (int k = 0; k < NF; ++k) {
    const double op = 1.0 + tau_L(k);
    if (k < e) {
      numer = numer * op;
    } else {
      Q = Q * sde_recip(op);
      A = A + tau * Q;
    }
  }
  const double U = K * A - (1.0 - Q), rn = sde_recip(numer);
  const double V = U > 0.0 ? U * rn : 0.0;
  if (GRAD) {
    const double itm = U > 0.0 ? rn : 0.0;
    double Qk = Q, tail = 0.0;  // Q_k, and sum_{j >= k} Q_j from the end
    // A one the compiler does not know to be the first loop's: it would keep that loop's 40 factors and their
    // reciprocals for this one, 160 registers, and spilled 180 of them in the f32 kernels.
    double one = 1.0;
    asm volatile("" : "+v"(one));
#pragma unroll
    for (int k = NF - 1; k >= 0; --k) {
      const double op = one + tau_L(k), x = (sizeof(R) == 4 ? tau : 1.0) * (double)H[k] * sde_recip(op);
      if (k < e) {
        M[k] = (R)(-V * x);
      } else {
        tail = tail + Qk;
        M[k] = (R)((-K * tau * tail - Q) * itm * x);
        Qk = Qk * op;
      }
    }
  }
  return V;
}

// The lane's Sobol entry and the wave's rows. Point index = path index; blocks of 256 make every wave one
// aligned run of 64 indices. Lane 0 has the wave's smallest index: if it is past the last path so is every
// lane of the wave, whose values are then never used.
__device__ __forceinline__ LmmSobol lmm_sobol(const LmmArgs& a, long long sid) {
  LmmSobol sb;
  const sde_u64 g = (sde_u64)sid ^ ((sde_u64)sid >> 1);
  sb.voff0 = (sde_u32)(g & 63u) * (sde_u32)(F * 4);
#pragma unroll
  for (int sl = 1; sl < NSL; ++sl) {
    const sde_u32 e = __builtin_amdgcn_readfirstlane((sde_u32)(g >> (6 + 8 * (sl - 1))) & 255u);
    sb.urow[sl - 1] = (sde_const_u32*)a.sobol_up + ((size_t)(sl - 1) * 256u + e) * (size_t)a.sobol_dims;
  }
  return sb;
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t lmm_sobol_rsrc(const LmmArgs& a) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)a.sobol_tab, (short)0, a.sobol_tab_words * 4, 0x00020000);
}

// MODE 0: price; 1: price and adjoint with checkpoints, the reverse sweep recomputing each
// segment into the segment tape; 2: the forward pass of the tape form, which writes every second state and
// L_N to the state tape and leaves the payoff, the reverse sweep and every partial to
// sdesim_lmm_reverse. The f32 checkpoint adjoint is held to 3 waves per SIMD (168 VGPRs): the
// extra wave hides the tape and LDS latency of its reverse sweep.
template <typename R, int MODE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(MODE == 1 && sizeof(R) == 4 ? 3 : 1)))
sdesim_lmm(const LmmArgs a) {
  constexpr int NQ = 2 + NF;
  if constexpr (sizeof(R) == 8) sde_normal_tab_load<R>(a.normal_tab);
  const long long S = a.paths;
  const int N = a.steps;
  const long long s = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = s < S;
  const long long sid = live ? s : 0;
  const sde_u32 voff = live ? (sde_u32)(sid * (long long)sizeof(R)) : 0x80000000u;

  const LmmSobol sb = lmm_sobol(a, sid);
  const __amdgpu_buffer_rsrc_t rsrc = lmm_sobol_rsrc(a);

  R Y[NF];
#pragma unroll
  for (int i = 0; i < NF; ++i) Y[i] = sizeof(R) == 4 ? R(0) : (R)((LmmDoubles)(sde_u64)a.tau_L0)[i];
  R* ck = (R*)a.checkpoints;
  int eta = 1, left = a.steps_per_period;  // n / steps_per_period + 1, without the division
  for (int n = 0; n < N; ++n) {
    if (MODE == 1 && (n % SEG) == 0 && live) {
      const long long slot = n / SEG;
#pragma unroll
      for (int i = 0; i < NF; ++i) ck[(slot * NF + i) * S + sid] = Y[i];
    }
    R eps[F];
    lmm_noise<R>(rsrc, sb, n, eps);
    if (MODE == 2 && (n & 1) == 0) {
      const SdeTapeSlot t = sde_tape_slot<R, NF>(a.tape, n >> 1, S);
      lmm_step<R>(lmm_rows<R>(a.rows), Y, eps, eta, [&](int i, R h) { sde_tape_put<R, 2>(t, voff, i, h); });
    } else {
      lmm_step<R>(lmm_rows<R>(a.rows), Y, eps, eta, [](int, R) {});
    }
    if (--left == 0) {
      left = a.steps_per_period;
      ++eta;
    }
  }
  R H[NF];
#pragma unroll
  for (int i = 0; i < NF; ++i) H[i] = lmm_held<R>(Y[i]);
  if (MODE == 2) {
    sde_tape_store<R, NF>(a.tape, (N + 1) >> 1, S, voff, H);
    return;
  }

  R M[NF];
  const double V = lmm_payoff<R, MODE == 1>(a, H, M);
  if constexpr (MODE == 1) {
    const R* tape = (const R*)a.tape;
    const int nseg = (N + SEG - 1) / SEG;
    for (int seg = nseg - 1; seg >= 0; --seg) {
      const int n0 = seg * SEG;
      const int len = N - n0 < SEG ? N - n0 : SEG;
#pragma unroll
      for (int i = 0; i < NF; ++i) Y[i] = ck[((long long)seg * NF + i) * S + sid];
      // H before steps n0 .. n0 + len - 2 go to the tape; the last stays in registers.
      for (int k = 0; k + 1 < len; ++k) {
        const SdeTapeSlot t = sde_tape_slot<R, NF>(a.tape, k, S);
        R eps[F];
        lmm_noise<R>(rsrc, sb, n0 + k, eps);
        lmm_step<R>(lmm_rows<R>(a.rows), Y, eps, (n0 + k) / a.steps_per_period + 1,
                    [&](int i, R h) { sde_tape_put<R, 0>(t, voff, i, h); });
      }
#pragma unroll
      for (int i = 0; i < NF; ++i) H[i] = lmm_held<R>(Y[i]);
      for (int k = len - 1; k >= 0; --k) {
        if (k + 1 < len) {
#pragma unroll
          for (int i = 0; i < NF; ++i) H[i] = tape[((long long)k * NF + i) * S + sid];
        }
        lmm_step_back<R>(lmm_rows<R>(a.rows_back), H, M, (n0 + k) / a.steps_per_period + 1);
      }
    }
  }
  sde_reduce_store_chunked<NQ>(
      [&](int q) { return !live ? 0.0 : q == 0 ? V : q == 1 ? V * V : MODE == 1 ? (double)M[q - 2] : 0.0; },
      a.partials + (long long)blockIdx.x * NQ);
}

// Reverse sweep of the tape form. H_N from the tape gives the payoff; then, two steps at a time from the
// last, A = H_n (n even) gives H_{n+1} in B, whose step back frees B for the tape's previous state while A's
// own step back runs (after step 0, step 0's again, unused). The next pair's normals are formed before that
// request: loads return in order, so their table words, asked for afterwards, would wait for the whole
// state. The f32 kernel is held to 3 waves per SIMD.
template <typename R>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sizeof(R) == 4 ? 3 : 1)))
sdesim_lmm_reverse(const LmmArgs a) {
  constexpr int NQ = 2 + NF;
  if constexpr (sizeof(R) == 8) sde_normal_tab_load<R>(a.normal_tab);
  const long long S = a.paths;
  const int N = a.steps;
  const long long s = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = s < S;
  const sde_u32 voff = live ? (sde_u32)(s * (long long)sizeof(R)) : 0x80000000u;

  const LmmSobol sb = lmm_sobol(a, live ? s : 0);
  const __amdgpu_buffer_rsrc_t rsrc = lmm_sobol_rsrc(a);

  R A[NF], B[NF], M[NF];
  sde_tape_load<R, NF>(a.tape, (N + 1) >> 1, S, voff, A);
  const double V = lmm_payoff<R, true>(a, A, M);
  int n = (N - 1) & ~1;
  R eps[F];
  lmm_noise<R>(rsrc, sb, n, eps);
  sde_tape_load<R, NF>(a.tape, n >> 1, S, voff, A);
  int eta = n / a.steps_per_period + 1, pos = n % a.steps_per_period;  // of step n; pos its place in its period
  for (; n >= 0; n -= 2) {
    if (n + 1 < N) {
      lmm_step_held<R>(lmm_rows<R>(a.rows), A, B, eps, eta);
      lmm_step_back<R>(lmm_rows<R>(a.rows_back), B, M, eta + (pos + 1 == a.steps_per_period ? 1 : 0));
    }
    const int before = n > 0 ? n - 2 : 0;
    lmm_noise<R>(rsrc, sb, before, eps);
    sde_tape_load<R, NF>(a.tape, before >> 1, S, voff, B);
    lmm_step_back<R>(lmm_rows<R>(a.rows_back), A, M, eta);
#pragma unroll
    for (int i = 0; i < NF; ++i) A[i] = B[i];
    for (pos -= 2; pos < 0; pos += a.steps_per_period) --eta;
  }
  sde_reduce_store_chunked<NQ>(
      [&](int q) { return !live ? 0.0 : q == 0 ? V : q == 1 ? V * V : (double)M[q - 2]; },
      a.partials + (long long)blockIdx.x * NQ);
}

}  // namespace

// mode: 0 price, 1 adjoint with checkpoints and the segment tape, 2 adjoint with the state tape
// (a.tape holds [(steps + 1) / 2 + 1][40][paths]; a forward and a reverse kernel).
hipError_t sdesim_launch_lmm(int f32, int mode, int grid, const LmmArgs& a, hipStream_t stream) {
#define SDE_LMM(R, MODE)                                                                                  \
  hipLaunchKernelGGL((sdesim_lmm<R, MODE>), dim3(grid), dim3(256), 0, stream, a);                            \
  if (MODE == 2) hipLaunchKernelGGL((sdesim_lmm_reverse<R>), dim3(grid), dim3(256), 0, stream, a);          \
  break;
  switch ((f32 ? 10 : 0) + mode) {
    case 12: SDE_LMM(float, 2)
    case 11: SDE_LMM(float, 1)
    case 10: SDE_LMM(float, 0)
    case 2: SDE_LMM(double, 2)
    case 1: SDE_LMM(double, 1)
    case 0: SDE_LMM(double, 0)
    default: return hipErrorInvalidValue;
  }
#undef SDE_LMM
  return hipGetLastError();
}
