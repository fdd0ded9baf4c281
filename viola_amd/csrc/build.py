"""Build libviola_hip.so for gfx950 with hipcc, and _host.so (the native host path) with the system compiler, in-tree next to
the sources.

python -m viola_amd.csrc.build        (or called by __graft_entry__.build())
"""

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

HERE = Path(__file__).resolve().parent
LIBRARY = HERE / "libviola_hip.so"
HOST_LIBRARY = HERE / "_host.so"                                          # Python extension: host.cpp over the C ABI
ARCH = "gfx950"
# -ffp-contract=off: the quantize / optimizer / codec kernels follow the reference's un-fused
# fp32 operation order so FP8 codes and scales come out bit-exact. The GEMM files apply their
# scale with an explicit fmaf.
COMMON = ["-O3", f"--offload-arch={ARCH}", "-fPIC", "-std=c++17", "-ffp-contract=off", "-fno-fast-math",
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-Wno-unused-command-line-argument"]
SOURCES = ["quantize.hip", "gemm.hip", "gemm_fast.hip", "gemm_fast_tensor.hip", "gemm_fast_mx.hip", "ns.hip", "ns_fast.hip", "optim.hip", "misc.hip", "tensor.hip"]


def hipcc():
    for candidate in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if candidate and (os.path.isabs(candidate) and os.path.exists(candidate) or not os.path.isabs(candidate)):
            return candidate
    raise RuntimeError("hipcc not found")


def _filter(text):
    return "\n".join(line for line in text.splitlines() if "is not a recognized feature for this target" not in line)


def _host_command():
    """host.cpp is host code only (autograd nodes, no kernels): the system compiler, torch's headers, the library above."""
    import sysconfig
    import torch
    from torch.utils.cpp_extension import include_paths
    torch_lib = Path(torch.__file__).parent / "lib"
    includes = [f"-I{path}" for path in include_paths("cuda")] + [f"-I{sysconfig.get_paths()['include']}"]
    return [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-w", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
            "-DTORCH_EXTENSION_NAME=_host", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *includes, str(HERE / "host.cpp"),
            "-o", str(HOST_LIBRARY), str(LIBRARY), f"-L{torch_lib}", "-ltorch_python", "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip",
            "-Wl,-rpath,$ORIGIN"]


def _build_host(incremental):
    sources = [HERE / "host.cpp", HERE.parents[1] / "include" / "viola_hip.h"]
    if incremental and HOST_LIBRARY.exists() and HOST_LIBRARY.stat().st_mtime > max(f.stat().st_mtime for f in sources):
        return
    result = subprocess.run(_host_command(), capture_output=True, text=True)
    if result.returncode != 0:
        raise RuntimeError("building the native host path failed:\n" + result.stdout + result.stderr)


def build(verbose=True, incremental=False):
    """Compile every source and link. incremental=True (a development convenience) reuses objects that
    are newer than their source and every header."""
    compiler = hipcc()
    objects = []
    newest_header = max(h.stat().st_mtime for h in HERE.glob("*.hpp"))

    def compile_one(name):
        obj = HERE / (name.rsplit(".", 1)[0] + ".o")
        if incremental and obj.exists() and obj.stat().st_mtime > newest_header and obj.stat().st_mtime > (HERE / name).stat().st_mtime:
            return obj
        cmd = [compiler, *COMMON, "-c", str(HERE / name), "-o", str(obj)]
        result = subprocess.run(cmd, capture_output=True, text=True)
        message = _filter(result.stdout + result.stderr)
        if result.returncode != 0:
            raise RuntimeError(f"hipcc failed for {name}:\n{message}")
        if verbose and message.strip():
            print(message, file=sys.stderr)
        return obj

    with ThreadPoolExecutor(max_workers=min(8, len(SOURCES))) as pool:
        objects = list(pool.map(compile_one, SOURCES))
    link = [compiler, f"--offload-arch={ARCH}", "-shared", "-fPIC", f"-Wl,-soname,{LIBRARY.name}", *map(str, objects), "-o", str(LIBRARY)]
    result = subprocess.run(link, capture_output=True, text=True)
    if result.returncode != 0:
        raise RuntimeError("link failed:\n" + _filter(result.stdout + result.stderr))
    _build_host(incremental)
    return LIBRARY


if __name__ == "__main__":
    print(build(incremental="--incremental" in sys.argv))
