"""Build libpscf_hip.so for gfx950 in-tree (pscf_amd/libpscf_hip.so).

    python -m pscf_amd.build
"""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

SOURCES = ["pscf_hip.hip", "am.cpp", "basis.cpp"]

HIP_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
    # no packed-FP32 instructions anywhere in the device code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # kernel arguments in scalar registers at wave start: a contour step is four
    # short kernels, and each began with a scalar load of its arguments
    # (gyroid 64^3 step 33.9 -> 32.7 us, BCC 32^3 18.6 -> 17.7 us)
    "-mllvm", "-amdgpu-kernarg-preload-count=10",
]


def build_lib(verbose=False, defines=None, out=None):
    """Compile the library; `defines` ({name: value}) set the build-time tuning
    knobs of the kernels (csrc/fft_lds.hpp and fft_reg.hpp: PSCF_LPV, the
    register-line factorisation variant; PSCF_ZLANES, lanes per z-column
    workgroup; PSCF_AJOBS, PSCF_ALIAS, PSCF_MAX_RADIX, PSCF_XPAD; and
    PSCF_TUNE_BUILD, only the autotuner's cubic lengths), `out` the output
    path."""
    srcs = [os.path.join(HERE, "csrc", f) for f in SOURCES]
    out = out or os.path.join(HERE, "libpscf_hip.so")
    tmp = out + ".tmp"
    dflags = ["-D%s=%s" % (k, v) for k, v in sorted((defines or {}).items())]
    cmd = [HIPCC] + HIP_FLAGS + dflags + srcs + ["-o", tmp]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("hipcc failed building libpscf_hip.so")
    os.replace(tmp, out)
    return out


FLANG = os.environ.get("FLANG", "/opt/rocm/lib/llvm/bin/flang")
FORTRAN_DIR = os.path.join(HERE, "fortran")
# dependency order of the drop-in modules
FORTRAN_MODULES = ["pscf_hip_c", "fft_mod", "chain_mod", "step_mod", "grid_basis_mod", "scf_mod"]


def build_fortran(verbose=False):
    """Compile the Fortran drop-in modules (pscf_amd/fortran) to objects and
    .mod files under pscf_amd/fortran/_build.  They `use` the reference's own
    kept modules (const_mod, grid_mod, basis_mod, chemistry_mod, ...), whose
    .mod files a driver build provides with -I; here only pscf_hip_c (the
    ISO_C_BINDING interface block) is compiled standalone, as a syntax check."""
    out = os.path.join(FORTRAN_DIR, "_build")
    os.makedirs(out, exist_ok=True)
    src = os.path.join(FORTRAN_DIR, "pscf_hip_c.f90")
    if not os.path.exists(src):
        return None
    cmd = [FLANG, "-O2", "-c", src, "-J", out, "-o", os.path.join(out, "pscf_hip_c.o")]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    return out


if __name__ == "__main__":
    print(build_lib(verbose=True))
    print(build_fortran(verbose=True))
