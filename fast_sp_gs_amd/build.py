"""Builds libfsgs_hip.so (hand-written HIP for gfx950) in-tree with hipcc, without any torch headers, and the native host
layer _host.so (C++ over torch's tensors and autograd, csrc/host) with the host compiler.

Every source is compiled to its own object (in parallel) and the objects are linked into one shared library.
`build()` recompiles everything; `build(incremental=True)` (or `python -m fast_sp_gs_amd.build -i`) recompiles only
sources that are newer than their object, or older than a header.
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
CSRC = PKG_DIR / "csrc"
OBJ_DIR = PKG_DIR / "build"
LIB_PATH = PKG_DIR / "libfsgs_hip.so"
HOST_SRC = CSRC / "host"
HOST_PATH = PKG_DIR / "_host.so"
HOST_SOURCES = ["torch_util.cpp", "surfel.cpp", "fast_surfel.cpp", "gaussian.cpp", "deform.cpp", "encode.cpp", "module.cpp"]
SOURCES = ["api.hip", "preprocess.hip", "binning.hip", "blend_fwd.hip", "blend_bwd.hip", "blend_topk.hip", "fast_preprocess.hip",
           "fast_blend.hip", "point_ops.hip", "knn_grid.hip", "lbs_bwd.hip", "ssim.hip", "epilogue.hip", "simple_knn.hip", "compaction.hip", "gs3d_preprocess.hip", "gs3d_blend.hip", "mlp.hip"]
HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fvisibility=hidden",
    # packed-FP32 instructions are kept out of the generated code on purpose
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]
NOISE = "packed-fp32-ops"


def hipcc_path() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if cand and (os.path.sep not in cand or os.path.exists(cand)):
            return cand
    return "hipcc"


def _host_flags():
    """(compile flags, link flags) of the host layer: torch's headers and libraries, the HIP runtime's headers."""
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths
    torch_lib = Path(torch.__file__).resolve().parent / "lib"
    compile_flags = ["-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
                     f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
                     *[f"-I{p}" for p in include_paths()], "-I/opt/rocm/include", f"-I{sysconfig.get_paths()['include']}"]
    link_flags = [f"-L{torch_lib}", "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip", f"-L{PKG_DIR}",
                  "-l:libfsgs_hip.so", "-Wl,-rpath,$ORIGIN"]
    return compile_flags, link_flags


def _run(cmd) -> str:
    proc = subprocess.run(cmd, capture_output=True, text=True)
    log = "\n".join(l for l in (proc.stdout + proc.stderr).splitlines() if NOISE not in l)
    if proc.returncode != 0:
        raise RuntimeError(f"compiler failed ({proc.returncode}): {' '.join(cmd)}\n{log}")
    return log


def build(verbose: bool = False, incremental: bool = False, jobs: int = 0) -> Path:
    """Compile every HIP source into one shared object, and the host layer that calls it into another."""
    OBJ_DIR.mkdir(exist_ok=True)
    hipcc = hipcc_path()
    headers_mtime = max(p.stat().st_mtime for p in list(CSRC.glob("*.hpp")) + list((PKG_DIR.parent / "include").glob("*.h")))
    cxx = os.environ.get("CXX", "g++")
    host_compile, host_link = _host_flags()
    host_mtime = max(headers_mtime, max(p.stat().st_mtime for p in HOST_SRC.glob("*.hpp")))
    todo = []  # (command, longest first: the host files take 20 s each)
    for s in HOST_SOURCES:
        src, obj = HOST_SRC / s, OBJ_DIR / (s + ".o")
        if not (incremental and obj.exists() and obj.stat().st_mtime > max(src.stat().st_mtime, host_mtime)):
            todo.append([cxx, *host_compile, "-c", str(src), "-o", str(obj)])
    for s in SOURCES:
        src, obj = CSRC / s, OBJ_DIR / (s + ".o")
        if not (incremental and obj.exists() and obj.stat().st_mtime > max(src.stat().st_mtime, headers_mtime)):
            todo.append([hipcc, *HIPCC_FLAGS, "-c", str(src), "-o", str(obj)])
    jobs = jobs or min(len(todo) or 1, int(os.environ.get("MAX_JOBS", os.cpu_count() or 4)), 16)
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        logs = list(pool.map(_run, todo))
    logs.append(_run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *[str(OBJ_DIR / (s + ".o")) for s in SOURCES],
                      "-o", str(LIB_PATH)]))
    logs.append(_run([cxx, "-shared", *[str(OBJ_DIR / (s + ".o")) for s in HOST_SOURCES], *host_link, "-o", str(HOST_PATH)]))
    if verbose:
        text = "\n".join(l for l in logs if l.strip())
        if text:
            print(text)
    return LIB_PATH


if __name__ == "__main__":
    print(build(verbose=True, incremental="-i" in sys.argv[1:]))
