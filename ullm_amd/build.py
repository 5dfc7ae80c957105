"""Build libullm_hip.so (the gfx950 kernels + C ABI) in-tree with hipcc.

Every translation unit under csrc/ is compiled for gfx950 only, in parallel,
then linked into ullm_amd/libullm_hip.so.  `python -m ullm_amd.build` or
`__graft_entry__.build()` runs it.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libullm_hip.so")
FRONT = os.path.join(HERE, "_front.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

# -packed-fp32-ops off: hipcc must not form v_pk_{add,mul,fma}_f32 on its own.
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-result",
]


def _sources():
    return sorted(
        os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith((".hip", ".cpp"))
    )


def _compile(src: str) -> str:
    obj = os.path.join(OBJ, os.path.basename(src) + ".o")
    cmd = [HIPCC, *FLAGS, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stderr}")
    return obj


def _build_front() -> None:
    """The native half of attention.py (csrc/front/front.cpp), host code only,
    against torch's headers and the library just built."""
    import sysconfig

    import torch

    t = os.path.dirname(torch.__file__)
    rocm = os.path.dirname(os.path.dirname(HIPCC))
    tmp = FRONT + ".tmp"
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           "-isystem", f"{t}/include", "-isystem", f"{t}/include/torch/csrc/api/include",
           "-isystem", f"{rocm}/include", "-isystem", sysconfig.get_paths()["include"],
           os.path.join(CSRC, "front", "front.cpp"), "-o", tmp, f"-L{HERE}", "-l:libullm_hip.so",
           f"-L{t}/lib", "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip",
           "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"front end failed:\n{r.stderr}")
    os.replace(tmp, FRONT)


def build(verbose: bool = True) -> str:
    """Compile every kernel source for gfx950, link libullm_hip.so, and build
    the front end on it."""
    os.makedirs(OBJ, exist_ok=True)
    srcs = _sources()
    jobs = min(len(srcs), int(os.environ.get("MAX_JOBS", "8")))
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(_compile, srcs))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", tmp]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    # Fail here, not on the GPU box, if a kernel stub or symbol went missing.
    import ctypes

    try:
        ctypes.CDLL(os.path.abspath(tmp))
    except OSError as e:
        raise RuntimeError(f"built library does not load: {e}") from None
    os.replace(tmp, LIB)
    _build_front()
    if verbose:
        print(f"built {LIB} from {len(srcs)} sources", file=sys.stderr)
    return LIB


if __name__ == "__main__":
    build()
