"""Build libzmoe_hip.so (the C-ABI MoE hot path) for gfx950 with hipcc, in-tree.

    python architecture-zarelga-superposition_amd/build_lib.py [-v] [--asan]

Objects go to ``_build/`` next to this file; the library to ``zmoe/libzmoe_hip.so``, and the
torch dispatcher kernels over it (csrc/eager_ops.cpp) to ``zmoe/libzmoe_eager.so``.
``--asan``: the host-sanitized build for the CPU tests, ``_build/asan/libzmoe_hip_asan.so``.
"""

from __future__ import annotations

import concurrent.futures as cf
import glob
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
INCLUDE = os.path.join(REPO, "include")
BUILD = os.path.join(HERE, "_build")
GEN = os.path.join(BUILD, "gen")
LIB = os.path.join(HERE, "zmoe", "libzmoe_hip.so")
EAGER_LIB = os.path.join(HERE, "zmoe", "libzmoe_eager.so")
ARCH = os.environ.get("ZMOE_OFFLOAD_ARCH", "gfx950")

# -packed-fp32-ops: never emit v_pk_{add,mul,fma}_f32 (the host pass warns that
# it does not know the feature; that is harmless).
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-result",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I", INCLUDE, "-I", CSRC, "-I", GEN,
]


def write_sigmoid_table(path: str) -> None:
    """The routing kernels' probability table: for each of the 65536 bf16 bit patterns z,
    the bf16 bits of sigmoid(z) evaluated in float64, rounded once to float32 and then to
    bf16 (round to nearest even); NaN logits give the quiet NaN 0x7fc0, and logits at or
    below -88.72283935546875 give 0 (torch's fp32 exp(-z) overflows there, so its sigmoid
    returns 0; the routing kernels' kSigmoidZeroBelow). Indexed by the
    logit's bits, it replaces a per-score exp when the gate's logits and its stored
    probabilities are bf16."""
    import numpy as np

    with np.errstate(all="ignore"):  # NaN patterns and exp overflow
        z = (np.arange(65536, dtype=np.uint32) << 16).view(np.float32).astype(np.float64)
        p = (1.0 / (1.0 + np.exp(-z))).astype(np.float32)
        p[z <= -88.72283935546875] = 0.0
    u = p.view(np.uint32).astype(np.uint64)
    bits = ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint32)
    bits[np.isnan(p)] = 0x7FC0
    rows = [", ".join(f"0x{b:04x}" for b in bits[i:i + 16]) for i in range(0, 65536, 16)]
    text = "// generated by build_lib.write_sigmoid_table; do not edit\n" + ",\n".join(rows) + "\n"
    old = open(path).read() if os.path.exists(path) else None
    if old != text:  # keep the file (and its timestamp) when unchanged
        with open(path, "w") as f:
            f.write(text)


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found")


# Host-only AddressSanitizer + UndefinedBehaviorSanitizer build of the same sources (the C-ABI
# shim's argument checks, workspace arithmetic and error reporting), for the CPU tests: each
# sanitizer flag applies to the host pass only, the device code is built as usual. Objects and
# the library go to _build/asan/; the library is loaded with the sanitizer runtime preloaded.
ASAN_BUILD = os.path.join(BUILD, "asan")
ASAN_LIB = os.path.join(ASAN_BUILD, "libzmoe_hip_asan.so")
ASAN_FLAGS = ["-Xarch_host", "-fsanitize=address,undefined", "-Xarch_host", "-fno-omit-frame-pointer",
              "-Xarch_host", "-fno-sanitize-recover=undefined", "-O1"]


def asan_runtime() -> str:
    """The clang AddressSanitizer runtime that hipcc's host compiler links against."""
    found = sorted(glob.glob(os.path.join(os.path.dirname(os.path.dirname(hipcc())), "llvm", "lib", "clang", "*",
                                          "lib", "linux", "libclang_rt.asan-x86_64.so")))
    if not found:
        raise RuntimeError("libclang_rt.asan-x86_64.so not found next to hipcc")
    return found[-1]


def _compile(src: str, verbose: bool, asan: bool = False) -> str:
    obj = os.path.join(ASAN_BUILD if asan else BUILD, os.path.basename(src).replace(".hip", ".o"))
    cmd = [hipcc(), *HIPCC_FLAGS, *(ASAN_FLAGS if asan else []), "-c", src, "-o", obj]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    msgs = [ln for ln in (res.stdout + res.stderr).splitlines() if "packed-fp32-ops" not in ln]
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n" + "\n".join(msgs))
    if verbose and msgs:
        print("\n".join(msgs), flush=True)
    return obj


def build(verbose: bool = False, jobs: int | None = None, asan: bool = False) -> str:
    os.makedirs(BUILD, exist_ok=True)
    os.makedirs(GEN, exist_ok=True)
    write_sigmoid_table(os.path.join(GEN, "zmoe_sigmoid_bf16.inc"))
    lib = ASAN_LIB if asan else LIB
    os.makedirs(os.path.dirname(lib), exist_ok=True)
    srcs = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    jobs = jobs or min(len(srcs), max(1, (os.cpu_count() or 4)))
    with cf.ThreadPoolExecutor(jobs) as ex:
        objs = list(ex.map(lambda s: _compile(s, verbose, asan), srcs))
    tmp = lib + ".tmp"
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs]
    if asan:  # the sanitizer runtime is preloaded by the process that loads this library
        cmd[2:2] = ["-Xarch_host", "-fsanitize=address,undefined", "-shared-libsan"]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("link failed:\n" + res.stdout + res.stderr)
    os.replace(tmp, lib)
    if not asan:
        build_eager_ops(verbose)
    return lib


def build_eager_ops(verbose: bool = False) -> str:
    """csrc/eager_ops.cpp (host code against torch's headers) into zmoe/libzmoe_eager.so, linked to
    the C ABI library next to it."""
    import torch
    from torch.utils import cpp_extension

    torch_lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    rocm = os.path.dirname(os.path.dirname(hipcc()))
    tmp = EAGER_LIB + ".tmp"
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-Wno-unused-function",
           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-I", INCLUDE,
           *(arg for path in cpp_extension.include_paths() for arg in ("-isystem", path)),
           "-isystem", os.path.join(rocm, "include"), os.path.join(CSRC, "eager_ops.cpp"), "-o", tmp,
           "-L", torch_lib, "-lc10", "-lc10_hip", "-ltorch_cpu", "-L", os.path.dirname(LIB), "-lzmoe_hip",
           "-Wl,-rpath,$ORIGIN"]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("eager ops failed to build:\n" + res.stdout + res.stderr)
    os.replace(tmp, EAGER_LIB)
    return EAGER_LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv, asan="--asan" in sys.argv))
