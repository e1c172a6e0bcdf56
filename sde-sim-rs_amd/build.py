"""Build libsdesim.so (gfx950) in-tree: sde_sim_rs/libsdesim.so.

Steps: embed the device headers (for hipRTC) and the Joe-Kuo D6 Sobol table (read from the
table scipy ships) into a generated source, compile the host runtime with g++, the
ahead-of-time kernels with hipcc for gfx950, and link. Run `python build.py` or call build().
"""
import concurrent.futures
import hashlib
import os
import subprocess
import sys

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
OUT = os.path.join(HERE, "sde_sim_rs", "libsdesim.so")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
HIPCC = os.path.join(ROCM, "bin", "hipcc")

# Packed FP32 instructions are disabled for every device compilation.
HIP_FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=fast",
             "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
HOST_FLAGS = ["-O2", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-function",
              "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROCM, "include")]

HOST_SOURCES = ["expr.cpp", "universe.cpp", "codegen.cpp", "runtime.cpp", "runtime_batch.cpp", "runtime_basket.cpp", "runtime_lmm.cpp"]
HIP_SOURCES = ["aot_kernels.hip", "batch_kernels.hip", "basket_kernels.hip", "lmm_kernels.hip"]


def _sobol_table():
    import scipy
    root = os.path.dirname(scipy.__file__)
    for rel in ("stats/_sobol_direction_numbers.npz", "stats/_qmc/_sobol_direction_numbers.npz"):
        path = os.path.join(root, rel)
        if os.path.exists(path):
            d = np.load(path)  # plain integer arrays; no pickle
            return d["poly"].astype(np.uint32), d["vinit"].astype(np.uint32)
    raise RuntimeError("scipy's Sobol direction-number table was not found")


def _ln_table():
    """[256][2] float64 (rc, 2 ln rc) for the device's -2 ln q: rc near 1 / c, c the middle of the
    j-th 256th of [1/2, 1), the one of 2^13 candidates whose 2 ln rc lies closest to a multiple of
    2^-45, which is what the second column holds (sums with multiples of -2 ln 2 are then exact)."""
    if np.finfo(np.longdouble).nmant < 63:
        raise RuntimeError("the logarithm table needs an extended-precision long double")
    mid = 0.5 * (1.0 + (np.arange(256) + 0.5) / 256.0)
    cand = (1.0 / mid)[:, None] + (np.arange(8192) - 4096)[None, :] * (1.1875 * 2.0 ** -42)
    v = 2 * np.log(cand.astype(np.longdouble)) * np.longdouble(2.0 ** 45)
    grid = np.floor(v + np.longdouble(0.5))
    off = np.abs(v - grid)
    best = np.argmin(off, axis=1)
    at = np.arange(256)
    if float(off[at, best].max()) > 1e-3:
        raise RuntimeError("no logarithm table within 1e-3 of the grid")
    return np.stack([cand[at, best], (grid[at, best] * np.longdouble(2.0 ** -45)).astype(np.float64)], axis=1)


def _batch_code_id():
    """16 hex digits of everything the batch kernels' code depends on: remembered launch configurations hold for it."""
    h = hashlib.sha256(" ".join(HIP_FLAGS).encode())
    for f in ("batch_kernels.hip", "reduce.hpp", "device/sdesim_device.hpp", "device/sdesim_args.hpp"):
        h.update(open(os.path.join(CSRC, f), "rb").read())
    h.update(_run([HIPCC, "--version"]).encode())
    return h.hexdigest()[:16]


def _raw(s, tag="SDEHDR"):
    assert (")" + tag + '"') not in s
    return 'R"' + tag + "(" + s + ")" + tag + '"'


def generate_embedded(path):
    with open(os.path.join(CSRC, "device", "sdesim_device.hpp")) as f:
        dev = f.read()
    with open(os.path.join(CSRC, "device", "sdesim_args.hpp")) as f:
        args = f.read()
    poly, vinit = _sobol_table()
    lines = ["// Generated by build.py: device headers for hipRTC and the Joe-Kuo D6 Sobol table.",
             'extern "C" {',
             'extern const char* sdesim_embedded_device_header;',
             'extern const char* sdesim_embedded_args_header;',
             'extern const int sdesim_jk_dims;',
             'extern const unsigned int sdesim_jk_poly[];',
             'extern const unsigned int sdesim_jk_vinit[];',
             'extern const double sdesim_ln_table[];',
             'extern const char* sdesim_batch_code_id;',
             'const char* sdesim_embedded_device_header = ' + _raw(dev) + ";",
             'const char* sdesim_embedded_args_header = ' + _raw(args) + ";",
             'const char* sdesim_batch_code_id = "' + _batch_code_id() + '";',
             'const int sdesim_jk_dims = %d;' % len(poly),
             'const unsigned int sdesim_jk_poly[] = {']
    lines.append(",".join(str(int(v)) for v in poly) + "};")
    lines.append('extern "C" const unsigned int sdesim_jk_vinit[] = {')
    flat = vinit.reshape(-1)
    for k in range(0, flat.size, 36):
        lines.append(",".join(str(int(v)) for v in flat[k:k + 36]) + ",")
    lines.append("};")
    lines.append('extern "C" const double sdesim_ln_table[] = {')
    lines.append(",".join(float(v).hex() for v in _ln_table().reshape(-1)) + "};")
    lines.append("}")
    text = "\n".join(lines) + "\n"
    old = open(path).read() if os.path.exists(path) else None
    if old != text:
        with open(path, "w") as f:
            f.write(text)


def _run(cmd):
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if r.returncode != 0:
        raise RuntimeError("command failed: %s\n%s" % (" ".join(cmd), r.stdout))
    return r.stdout


def build(verbose=False):
    os.makedirs(BUILD, exist_ok=True)
    emb = os.path.join(BUILD, "embedded.cpp")
    generate_embedded(emb)
    jobs = []
    objs = []
    for src in HOST_SOURCES:
        obj = os.path.join(BUILD, src + ".o")
        jobs.append(["g++"] + HOST_FLAGS + ["-c", os.path.join(CSRC, src), "-o", obj])
        objs.append(obj)
    obj = os.path.join(BUILD, "embedded.o")
    jobs.append(["g++", "-O0", "-fPIC", "-c", emb, "-o", obj])
    objs.append(obj)
    for src in HIP_SOURCES:
        obj = os.path.join(BUILD, src + ".o")
        jobs.append([HIPCC] + HIP_FLAGS + ["-c", os.path.join(CSRC, src), "-o", obj])
        objs.append(obj)
    with concurrent.futures.ThreadPoolExecutor(max_workers=min(8, len(jobs))) as ex:
        for out in ex.map(_run, jobs):
            if verbose and out.strip():
                print(out)
    tmp = OUT + ".tmp"
    _run([HIPCC, "-shared", "-fPIC", "--offload-arch=gfx950", "-o", tmp] + objs +
         ["-L" + os.path.join(ROCM, "lib"), "-lhiprtc", "-lamdhip64", "-Wl,-rpath," + os.path.join(ROCM, "lib")])
    os.replace(tmp, OUT)
    return OUT


# Host-side sanitizers for the CPU build of the runtime (parser, code generator, Sobol tables, ABI
# checks). The device code is not built with them: the ahead-of-time kernel objects are the
# regular ones, and the library is linked by g++.
SANITIZE_FLAGS = ["-fsanitize=address,undefined", "-fno-sanitize-recover=undefined", "-fno-omit-frame-pointer", "-g"]


def build_sanitized(out_path):
    """libsdesim.so with AddressSanitizer and UndefinedBehaviorSanitizer in the host runtime, written
    to `out_path` (load it with the sanitizer runtimes preloaded: see sanitizer_env)."""
    build()  # the regular objects, including the ahead-of-time kernels
    sb = os.path.join(BUILD, "sanitized")
    os.makedirs(sb, exist_ok=True)
    flags = [f for f in HOST_FLAGS if f != "-O2"] + ["-O1"] + SANITIZE_FLAGS
    jobs, objs = [], []
    for src in HOST_SOURCES:
        obj = os.path.join(sb, src + ".o")
        jobs.append(["g++"] + flags + ["-c", os.path.join(CSRC, src), "-o", obj])
        objs.append(obj)
    with concurrent.futures.ThreadPoolExecutor(max_workers=min(8, len(jobs))) as ex:
        list(ex.map(_run, jobs))
    objs.append(os.path.join(BUILD, "embedded.o"))
    objs += [os.path.join(BUILD, src + ".o") for src in HIP_SOURCES]
    _run(["g++", "-shared", "-o", out_path] + objs + SANITIZE_FLAGS +
         ["-L" + os.path.join(ROCM, "lib"), "-lhiprtc", "-lamdhip64", "-Wl,-rpath," + os.path.join(ROCM, "lib")])
    return out_path


def sanitizer_env(env=None):
    """Environment for a Python process that loads the sanitized library: the ASan and UBSan
    runtimes preloaded (the interpreter itself is not instrumented), leak checking off (the
    interpreter's own allocations at exit), every report fatal."""
    env = dict(os.environ if env is None else env)
    libs = []
    for name in ("libasan.so", "libubsan.so"):
        libs.append(subprocess.run(["g++", "-print-file-name=" + name], stdout=subprocess.PIPE, text=True,
                                   check=True).stdout.strip())
    env["LD_PRELOAD"] = " ".join(libs + ([env["LD_PRELOAD"]] if env.get("LD_PRELOAD") else []))
    env["ASAN_OPTIONS"] = "detect_leaks=0:abort_on_error=1:halt_on_error=1"
    env["UBSAN_OPTIONS"] = "print_stacktrace=1:halt_on_error=1"
    return env


if __name__ == "__main__":
    print(build(verbose=True))
