"""Builds the HIP shared library libbeep_gpu.so in-tree for gfx950.

The library holds the device kernels, the C ABI of include/beep_gpu.h and the
C++ host model (normalisation and parameter-derived tables)."""
import hashlib
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libbeep_gpu.so")
SOURCES = ["beep_gpu.hip", "host_model.cc", "host/gpu_state.cc"]
HEADERS = ["device_rng.hh", "fused_common.hh", "fused_spec.hh", "step_spec.hh", "kernels.hh", "obs_kernels.hh", "pmcmc_kernels.hh", "replay_kernels.hh",
           "step_kernels.hh", "host_model.hh", "host/gpu_state.hh"]
# Headers the library compiles at run time (hiprtc) for each compartment
# structure, embedded as string constants.
JIT_HEADERS = [("kJitDeviceRng", "device_rng.hh"), ("kJitFusedCommon", "fused_common.hh"),
               ("kJitFusedSpec", "fused_spec.hh"), ("kJitStepSpec", "step_spec.hh")]
# The fused kernels, generic and specialised: what tuned workgroup sizes hold for.
TUNED_SOURCES = ["device_rng.hh", "fused_common.hh", "fused_spec.hh", "kernels.hh"]
JIT_INC = os.path.join(CSRC, "jit_sources.inc")
# Compartment structures the run-time compiled kernel is checked with at build
# time: SEIR (S->E, E->I, I->R, I infectious) with one strain, and the same
# with two strains (which compiles the pooling of susceptibles).
CHECK_PRELUDES = ["""#define BEEP_SPEC_FUSED
#define BEEP_SPEC_REPLAY
#define BEEP_SPEC_STEP
namespace beepspec {
constexpr int C = 4, T = 3, G = %d, CP = 4, INF_TR = 0, MIN_WAVES = 4, STEP_WAVES = 4, NSTRAIN = %d, DPM = 1;
constexpr bool GROUPED = %s, N_TV = false, MODS = false, AF_STATIC = true, STAGED = true, Q16 = true;
constexpr bool KEEP_TN = true, KEEP_TM = true, KEEP_PT = true;
constexpr int FROM[3] = {0, 1, 2};
constexpr int TO[3] = {1, 2, 3};
constexpr bool INFC[4] = {false, false, true, false};
}  // namespace beepspec
""" % (g, g, "true" if g == 2 else "false") for g in (1, 2)]
CHECK_SRC = os.path.join(CSRC, "host", "gpu_state_check.cc")
CHECK_BIN = os.path.join(HERE, "bin", "gpu_state_check")


def hipcc():
    for p in ("/opt/rocm/bin/hipcc", "hipcc"):
        if os.path.sep not in p or os.path.exists(p):
            return p
    return "hipcc"


def write_jit_sources():
    """jit_sources.inc: the run-time compiled headers as raw string literals,
    and a tag of the fused kernels' sources, under which tuned workgroup sizes
    are saved."""
    out = ["// Generated by beep_amd/build.py from the headers named below; do not edit.\n"]
    for name, fn in JIT_HEADERS:
        text = open(os.path.join(CSRC, fn)).read()
        if ")BEEPJIT\"" in text:
            raise RuntimeError(f"{fn} contains the raw-string delimiter")
        out.append(f"static const char {name}[] = R\"BEEPJIT({text})BEEPJIT\";\n")
    tag = hashlib.sha256("".join(open(os.path.join(CSRC, fn)).read() for fn in TUNED_SOURCES).encode()).hexdigest()[:16]
    out.append(f"static const char kKernelTag[] = \"{tag}\";\n")
    tmp = JIT_INC + ".tmp"
    with open(tmp, "w") as f:
        f.write("".join(out))
    os.replace(tmp, JIT_INC)


def check_spec_kernel(verbose=True):
    """Compiles the structure-specialised kernel ahead of time for one
    structure, so that a compile error shows at build time rather than when a
    context is created."""
    import tempfile
    for prelude in CHECK_PRELUDES:
        _check_one(prelude, verbose)


def _check_one(prelude, verbose):
    import tempfile
    with tempfile.TemporaryDirectory() as d:
        src = os.path.join(d, "spec_check.hip")
        with open(src, "w") as f:
            f.write(prelude + '#include "fused_common.hh"\n#include "fused_spec.hh"\n#include "step_spec.hh"\n')
        cmd = [hipcc(), "--offload-arch=gfx950", "-O3", "-std=c++17", "--cuda-device-only", "-c",
               "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-I", CSRC, "-o",
               os.path.join(d, "spec_check.o"), src]
        if verbose:
            print(" ".join(cmd), flush=True)
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            sys.stderr.write(r.stdout + r.stderr)
            raise RuntimeError("the structure-specialised kernel does not compile")


def build(verbose=True):
    """Compiles every source for gfx950 and links libbeep_gpu.so.  Always
    recompiles (the build check must exercise the compiler)."""
    write_jit_sources()
    check_spec_kernel(verbose)
    cmd = [hipcc(), "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
           "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
           "-Wall", "-Wno-unused-function", "-Wno-unused-variable",
           "-I", os.path.join(ROOT, "include"),
           "-o", LIB + ".tmp"] + [os.path.join(CSRC, s) for s in SOURCES] + ["-lhiprtc"]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("hipcc failed building libbeep_gpu.so")
    os.replace(LIB + ".tmp", LIB)
    # The C++ host mirror's self-check program, linked against the library.
    os.makedirs(os.path.dirname(CHECK_BIN), exist_ok=True)
    cmd = [hipcc(), "-O2", "-std=c++17", "-I", os.path.join(ROOT, "include"), "-I", os.path.join(CSRC, "host"),
           CHECK_SRC, "-o", CHECK_BIN + ".tmp", "-L", HERE, "-lbeep_gpu", "-Wl,-rpath,$ORIGIN/.."]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("building gpu_state_check failed")
    os.replace(CHECK_BIN + ".tmp", CHECK_BIN)
    return LIB


if __name__ == "__main__":
    build()
