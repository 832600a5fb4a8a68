"""Build ``libti8.so`` (every HIP kernel + the C ABI) for gfx950 with hipcc, and the layer call's host side with g++.

Run as ``python triton-int8_amd/build.py`` or call :func:`build`.  The libraries are
written next to this file; it is cross-compiled, so no GPU is needed to build.
"""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libti8.so")
NATIVE = os.path.join(HERE, "_native.so")
SOURCES = ["api.hip", "quant.hip", "fwht.hip", "gemm.hip", "gemm_chain.hip", "gemm_mid.hip", "gemm_skinny.hip", "gemm_decode.hip", "step.hip", "decoder.hip", "attention.hip", "bias.hip", "probe.hip"]

# -ffp-contract=off: x*scale+0.5 must round twice (bit-exact quantisation); kernels
#   that want an fma ask for one explicitly.
# -packed-fp32-ops disabled: keep hipcc from forming v_pk_*_f32 from scalar float code.
# -amdgpu-mfma-vgpr-form: MFMA accumulators in ordinary VGPRs, so the block-channel promotion
#   (convert + fma on every 128-deep partial) reads them without v_accvgpr_read copies.
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-Wno-unused-command-line-argument",
         "-mllvm", "-amdgpu-mfma-vgpr-form"]


def build(verbose: bool = False) -> str:
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    cmd = [hipcc] + FLAGS + ["-o", LIB] + [os.path.join(CSRC, s) for s in SOURCES]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in res.stdout.splitlines() if "packed-fp32-ops" not in l and l.strip())
    if res.returncode != 0:
        raise RuntimeError("hipcc failed:\n" + out)
    if verbose and out:
        print(out)
    try:
        build_native(verbose)
    except (OSError, RuntimeError, ImportError) as e:      # no g++, no headers of torch or Python: the layer calls are then made from Python
        if os.path.exists(NATIVE):
            os.remove(NATIVE)
        print(f"{NATIVE} was not built, layer calls take the Python way: {e}", file=sys.stderr, flush=True)
    return LIB


def build_native(verbose: bool = False) -> str:
    """The layer call's host side (csrc/native.cpp), an extension of the Python and the torch that run this: host code only, it is
    handed the library's entry points when it is loaded."""
    import sysconfig
    import torch
    from torch.utils.cpp_extension import include_paths, library_paths
    # NDEBUG: without it pybind11's headers put a thread-local counter into the library, and once a library with thread-local storage that
    # nobody touches has been loaded, glibc looks every other thread-local variable up the long way (torch's calls take 10 to 20 % longer)
    cmd = ["g++", "-O2", "-DNDEBUG", "-std=c++17", "-fPIC", "-shared", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}",
           f'-DTI8_BUILT_FOR_TORCH="{torch.__version__}"']
    cmd += [a for path in [sysconfig.get_paths()["include"], *include_paths()] for a in ("-isystem", path)]
    cmd += [os.path.join(CSRC, "native.cpp"), "-o", NATIVE, *(f"-L{path}" for path in library_paths()), "-ltorch_python", "-ltorch_cpu", "-lc10"]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if res.returncode != 0:
        raise RuntimeError("g++ failed:\n" + res.stdout)
    return NATIVE


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
