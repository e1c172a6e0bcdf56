// runtime_basket.cpp -- host side of the correlated-basket price / adjoint kernels
// (include/sdesim.h: sdesim_basket_*). No reference counterpart: the reference computes no
// sensitivities; a basket in the reference is a universe of correlated GBM equations whose
// Cholesky factors are written into the coefficients.
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "../../include/sdesim.h"
#include "device/sdesim_args.hpp"

hipError_t sdesim_launch_basket(int f32, int assets, int adjoint, int team, int again, int grid, const BasketArgs& a,
                                int nq, double* sums, hipStream_t stream);
hipError_t sdesim_normal_table(int f32, const void** out);
int sdesim_set_error(int code, const std::string& msg);
void sdesim_log(const char* fmt, ...);

namespace {
struct BFail {
  int code;
  std::string msg;
};
void bk(hipError_t e, const char* what) {
  if (e != hipSuccess) throw BFail{SDESIM_ERUNTIME, std::string(what) + ": " + hipGetErrorString(e)};
}
template <class F>
int guard(F&& f) {
  try {
    f();
    return SDESIM_OK;
  } catch (const BFail& e) {
    return sdesim_set_error(e.code, e.msg);
  } catch (const std::exception& e) {
    return sdesim_set_error(SDESIM_ERUNTIME, e.what());
  }
}
}  // namespace

struct sdesim_basket {
  sdesim_basket_spec spec{};
  int nq = 0;         // reduced quantities of the adjoint
  long long grid = 0;
  bool team = false;  // blocks of four waves to 64 paths (few paths), else a path per lane
  int storage = SDESIM_STORAGE_CHECKPOINTS;  // as asked for, or AUTO's choice; neither keeps states
  double* partials = nullptr;
  double* sums = nullptr;
  const void* normal_tab = nullptr;         // the device's shared table of the inverse normal
  ~sdesim_basket() {
    if (partials) (void)hipFree(partials);
    if (sums) (void)hipFree(sums);
  }
};

extern "C" {

int sdesim_basket_create(const sdesim_basket_spec* spec, sdesim_basket** out) {
  return guard([&] {
    if (!spec || !out) throw BFail{SDESIM_EVALUE, "null argument"};
    const sdesim_basket_spec& s = *spec;
    if (s.assets < 1 || s.assets > 8) throw BFail{SDESIM_EVALUE, "assets must be between 1 and 8"};
    if (s.steps < 1) throw BFail{SDESIM_EVALUE, "steps must be >= 1"};
    if (s.paths < 1) throw BFail{SDESIM_EVALUE, "paths must be >= 1"};
    if (!(s.horizon > 0.0)) throw BFail{SDESIM_EVALUE, "horizon must be > 0"};
    if (!(s.width >= 0.0)) throw BFail{SDESIM_EVALUE, "width must be >= 0"};
    if (s.storage < SDESIM_STORAGE_AUTO || s.storage > SDESIM_STORAGE_CHECKPOINTS)
      throw BFail{SDESIM_EVALUE, "storage must be SDESIM_STORAGE_AUTO, _TAPE or _CHECKPOINTS"};
    std::unique_ptr<sdesim_basket> b(new sdesim_basket());
    b->spec = s;
    // Teams up to two blocks per CU (32,768 paths): 0.225 instead of 0.30 ms for a call there (8 assets with Greeks,
    // f64, 100 steps); at twice as many paths they gain nothing (0.32 against 0.29).
    int dev = 0, cus = 0;
    bk(hipGetDevice(&dev), "hipGetDevice");
    bk(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev), "hipDeviceGetAttribute");
    const long long waves = (s.paths + 63) / 64;
    b->team = waves <= 2LL * cus;
    b->grid = b->team ? waves : (s.paths + 255) / 256;
    if (b->grid > 0x7fffffffLL) throw BFail{SDESIM_EVALUE, "too many paths"};
    // The derivatives are summed on the way forward: no state is stored under either name. What a tape
    // was refused for, a step of it (at 1 or 8 assets) of 2^31 bytes or more, still is.
    const size_t rb = s.precision == SDESIM_F32 ? 4 : 8;
    const bool tape_addressable = (size_t)(s.assets == 1 ? 1 : 8) * (size_t)s.paths * rb < (1ull << 31);
    if (s.storage == SDESIM_STORAGE_TAPE && !tape_addressable)
      throw BFail{SDESIM_EVALUE, "the tape needs assets * paths * size < 2^31 bytes per step"};
    if (s.storage != SDESIM_STORAGE_CHECKPOINTS && tape_addressable) b->storage = SDESIM_STORAGE_TAPE;
    b->nq = 2 + 3 * s.assets + s.assets * (s.assets + 1) / 2;
    bk(sdesim_normal_table(s.precision == SDESIM_F32 ? 1 : 0, &b->normal_tab), "inverse normal table");
    bk(hipMalloc(&b->partials, sizeof(double) * b->nq * b->grid), "hipMalloc(partials)");
    bk(hipMalloc(&b->sums, sizeof(double) * b->nq), "hipMalloc(sums)");
    sdesim_log("basket: %d assets, %lld paths, %d steps", s.assets, (long long)s.paths, s.steps);
    *out = b.release();
  });
}

void sdesim_basket_free(sdesim_basket* b) { delete b; }

int32_t sdesim_basket_storage(const sdesim_basket* b) { return b ? b->storage : -1; }

int sdesim_basket_eval(sdesim_basket* b, const double* x0, const double* mu, const double* sigma,
                       const double* weight, const double* chol, int32_t adjoint, double* out, void* stream) {
  return guard([&] {
    if (!b || !x0 || !mu || !sigma || !weight || !chol || !out) throw BFail{SDESIM_EVALUE, "null argument"};
    const sdesim_basket_spec& s = b->spec;
    const int A = s.assets;
    BasketArgs a;
    std::memset(&a, 0, sizeof a);
    a.dt = s.horizon / s.steps;
    a.sdt = std::sqrt(a.dt);
    for (int i = 0; i < A; ++i) {
      a.x0[i] = x0[i];
      a.sigma[i] = sigma[i];
      a.weight[i] = weight[i];
      a.mdt[i] = mu[i] * a.dt;
      a.mdt_f[i] = (float)a.mdt[i];
      for (int k = 0; k <= i; ++k) {
        const int q = i * 8 + k;
        a.chol[q] = chol[i * A + k];
        a.scl[q] = sigma[i] * a.sdt * a.chol[q];
        a.scl_f[q] = (float)a.scl[q];
      }
    }
    a.strike = s.strike;
    a.width = s.width;
    a.seed = s.seed;
    a.paths = s.paths;
    a.steps = s.steps;
    a.partials = b->partials;
    a.normal_tab = b->normal_tab;
    hipStream_t st = (hipStream_t)stream;
    const int nq = adjoint ? b->nq : 2;
    std::vector<double> sums(nq);
    auto run = [&](int again) {
      bk(sdesim_launch_basket(s.precision == SDESIM_F32 ? 1 : 0, A, adjoint != 0, b->team, again, (int)b->grid, a, nq,
                              b->sums, st),
         "basket launch");
      bk(hipMemcpyAsync(sums.data(), b->sums, sizeof(double) * nq, hipMemcpyDeviceToHost, st), "hipMemcpyAsync");
      bk(hipStreamSynchronize(st), "hipStreamSynchronize");
    };
    run(0);
    // Derivatives that are not finite: a path with a growth factor of 0 (or inputs that give no others).
    if (adjoint && !std::all_of(sums.begin() + 2, sums.end(), [](double v) { return std::isfinite(v); })) run(1);
    const double n = (double)s.paths;
    const double m1 = sums[0] / n;
    out[0] = m1;
    out[1] = s.paths > 1 ? (sums[1] - sums[0] * m1) / (n - 1.0) : 0.0;
    if (adjoint)
      for (int q = 2; q < nq; ++q) out[q] = sums[q] / n;
  });
}

}  // extern "C"
