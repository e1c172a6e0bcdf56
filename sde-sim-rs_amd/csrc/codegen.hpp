// codegen.hpp -- HIP source for one universe + options (compiled at run time with hipRTC).
#pragma once
#include <string>
#include <vector>

#include "universe.hpp"

// In a generated function body: products are fused into sums of their own statement only. Sources that have it are
// compiled with the option under which clang honours it.
#define SDE_FUSE_IN_STATEMENTS "#pragma clang fp contract(on)"

namespace sdesim {

struct CodegenOptions {
  int scheme = 0;       // 0 Euler-Maruyama, 1 "Runge-Kutta first order"
  int compat = 0;       // 0 reference cache semantics, 1 textbook (refresh from settled rows)
  bool f32 = false;     // f32 state and coefficients (f64 uniforms and estimator sums)
  int rng = 0;          // SDE_RNG_* in sdesim_device.hpp
  int out = 1;          // SDE_OUT_* bit mask
  int ppl = 1;          // paths per lane
  int block = 256;      // threads per block
  int nsl = 1;          // Sobol table slices (Gray-code bits covered: 6 + 8 (nsl - 1))
  bool uniform_grid = false;  // every dt and sqrt(dt) is bitwise equal in the kernel's precision
  bool wave_aligned = false;  // Sobol index of path 0 is a multiple of 64 and blocks hold whole waves
  int team = 1;         // waves to 64 paths: 1 = sde_path_kernel, else sde_team_kernel
  bool library_f64 = false;   // f64: library logarithm and roots (reaches_root below)
  bool steps = true;    // false when the time grid has a single point (nothing is evaluated)
  std::string payoff;   // expression over process names and t at the last time point
  std::string name = "sdesim_kernel";  // entry point name
};

struct UndefinedName : std::runtime_error {
  using std::runtime_error::runtime_error;
};

// A condition under which the reference panics (surfaced by PyO3 as PanicException).
struct Panic : std::runtime_error {
  using std::runtime_error::runtime_error;
};

// Returns the complete kernel source (entry point `o.name`). Throws ParseError for a bad
// payoff, UndefinedName when an evaluated expression names an unknown variable, and
// Panic for the reference's run-time panics (RK with no stochastic increment).
std::string generate_kernel_source(const Universe& u, const CodegenOptions& o);

// Descriptive entry point name: sdesim_<em|rk>_<f32|f64>_<rng>_<filt|term|filt_term>.
std::string kernel_name(const CodegenOptions& o);

// Whether the noise of the universe holds a root that may let rounding differences grow. With noise s sqrt(x)
// and drift a at x = 0, an Euler path that steps out of 0 lands at about a dt, where its next increment changes
// by s sqrt(dt) / (2 sqrt(a dt)) = s / (2 sqrt(a)) of any difference: above 1, two copies of a path that
// differ in one last bit drift apart without bound (CIR with 4 a / s^2 = 0.18: 0.1 apart after 1550 steps),
// below 1 they come together (Heston's variance at 1.28: 1e-15 after 1024). Any other root has such a place too,
// wherever its argument vanishes (0.8 sqrt(x (1 - x)) at 1 with a drift of 0.015 to it: 0.67 after 1550). So the
// only roots of a Levy process in a noise coefficient that are taken to be harmless are those of a process x, or
// max(x, 0), whose own drift and noise depend on x alone and at 0 have 4 a >= s^2, or noise that vanishes like x
// itself and a >= 0 (a geometric variance: differences stay in proportion to it); every other power below 1,
// logarithm or inverse function counts. The f64 kernels of such universes, and the batch kernel's CIR
// instances with 4 a < s^2, keep the library's logarithm, root and division, so that their paths stay bit for bit
// those of the general inverse normal.
bool reaches_root(const Universe& u);

}  // namespace sdesim
