"""Builds libelyhip.so, the gfx950 code object of this package, in-tree.

    python -m elysium_wan_amd.build        # or __graft_entry__.build()

Every csrc/*.hip translation unit is compiled by hipcc for gfx950 only and
linked into elysium_wan_amd/libelyhip.so, which the package loads with ctypes.
csrc/binding.cpp (host code against torch's headers) becomes
elysium_wan_amd/_native.so beside it, the plain calls' way into that library.
Flags that matter for the numerics:

* -ffp-contract=off: no fused multiply-add unless the source writes one, so
  HostAdamW's one-rounding-per-op sequence survives compilation.
* -fhip-fp32-correctly-rounded-divide-sqrt: IEEE fp32 division and sqrt.
* -fno-gpu-flush-denormals-to-zero: fp32 subnormals are kept, as on the CPU.
* -Xclang -target-feature -Xclang -packed-fp32-ops: no packed fp32 ALU ops
  (v_pk_{add,mul,fma}_f32) in any kernel; the host pass warns that it does
  not know the feature, which is harmless.
"""

from __future__ import annotations

import concurrent.futures as cf
import glob
import os
import shutil
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libelyhip.so")
NATIVE = os.path.join(HERE, "_native.so")
ARCH = "gfx950"

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fno-gpu-rdc",
    "-ffp-contract=off",
    "-fhip-fp32-correctly-rounded-divide-sqrt",
    "-fno-gpu-flush-denormals-to-zero",
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-function",
]


def hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(path):
        raise RuntimeError("hipcc not found: the HIP library cannot be built")
    return path


def _compile(src: str) -> str:
    obj = os.path.join(BUILD, os.path.basename(src) + ".o")
    cmd = [hipcc(), *HIPCC_FLAGS, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{r.stdout}\n{r.stderr}")
    return obj


def _compile_native() -> str:
    """csrc/binding.cpp to an object file, with the host compiler."""
    import torch

    obj = os.path.join(BUILD, "binding.cpp.o")
    inc = os.path.join(os.path.dirname(torch.__file__), "include")
    cmd = [
        "g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
        f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
        f"-I{inc}", f"-I{os.path.join(inc, 'torch', 'csrc', 'api', 'include')}", f"-I{sysconfig.get_paths()['include']}",
        f"-I{os.path.join(os.environ.get('ROCM_PATH', '/opt/rocm'), 'include')}",
        "-c", os.path.join(CSRC, "binding.cpp"), "-o", obj,
    ]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed on binding.cpp:\n{r.stdout}\n{r.stderr}")
    return obj


def _link_native(obj: str) -> None:
    import torch

    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    tmp = NATIVE + ".tmp"
    cmd = ["g++", "-shared", "-o", tmp, obj, f"-L{HERE}", "-lelyhip", f"-L{lib}", "-lc10", "-lc10_hip", "-ltorch_cpu",
           "-ltorch_hip", "-ltorch", "-ltorch_python", "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link of _native.so failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, NATIVE)


def build(verbose: bool = False) -> str:
    """Compile every csrc/*.hip for gfx950 and link libelyhip.so, then
    _native.so against it (always rebuilds).  Returns the library path."""
    os.makedirs(BUILD, exist_ok=True)
    srcs = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    if not srcs:
        raise RuntimeError(f"no HIP sources under {CSRC}")
    jobs = min(len(srcs), max(1, min(8, os.cpu_count() or 1)))
    with cf.ThreadPoolExecutor(jobs) as ex:
        native = ex.submit(_compile_native)
        objs = list(ex.map(_compile, srcs))
    tmp = LIB + ".tmp"
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    _link_native(native.result())
    if verbose:
        print(f"built {LIB} from {len(srcs)} sources", file=sys.stderr)
    return LIB


if __name__ == "__main__":
    build(verbose=True)
