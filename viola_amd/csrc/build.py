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
SOURCES = ["gemm_generic.hip", "gemm_fast.hip", "gemm_fast_mx.hip", "gemm_fast_tensor.hip", "gemm_pingpong_grouped.hip", "gemm_pingpong_mx.hip", "gemm_pingpong_tensor.hip", "gemm.hip", "gemm_skinny.hip", "quantize.hip", "ns.hip", "ns_fast.hip", "optim.hip", "misc.hip", "tensor.hip"]


def hipcc():
    for candidate in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if candidate and (os.path.isabs(candidate) and os.path.exists(candidate) or not os.path.isabs(candidate)):
            return candidate
    raise RuntimeError("hipcc not found")


def _filter(text):
    return "\n".join(line for line in text.splitlines() if "is not a recognized feature for this target" not in line)


HOST_SOURCES = ["host.cpp", "host_optim.cpp"]


def _host_flags():
    """Host code only (autograd nodes, no kernels): the system compiler, torch's headers, the library above."""
    import sysconfig
    import torch
    from torch.utils.cpp_extension import include_paths
    torch_lib = Path(torch.__file__).parent / "lib"
    includes = [f"-I{path}" for path in include_paths("cuda")] + [f"-I{sysconfig.get_paths()['include']}"]
    compile_flags = ["-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-w", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-DTORCH_EXTENSION_NAME=_host",
                     f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *includes]
    link_flags = ["-shared", str(LIBRARY), f"-L{torch_lib}", "-ltorch_python", "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip", "-Wl,-rpath,$ORIGIN"]
    return compile_flags, link_flags


def _run(command, what):
    result = subprocess.run(command, capture_output=True, text=True)
    if result.returncode != 0:
        raise RuntimeError(f"{what} failed:\n" + _filter(result.stdout + result.stderr))


def _host_object(name, incremental):
    obj, headers = HERE / (name.rsplit(".", 1)[0] + ".o"), [HERE / "host.hpp", HERE.parents[1] / "include" / "viola_hip.h"]
    if not (incremental and obj.exists() and obj.stat().st_mtime > max(f.stat().st_mtime for f in [HERE / name, *headers])):
        _run([os.environ.get("CXX", "g++"), *_host_flags()[0], "-c", str(HERE / name), "-o", str(obj)], f"compiling {name}")
    return obj


def build(verbose=True, incremental=False):
    """Compile every source and link. incremental=True (a development convenience) reuses objects that
    are newer than their source and every header."""
    compiler = hipcc()
    objects = []
    newest_header = max(h.stat().st_mtime for h in HERE.glob("*.hpp") if h.name != "host.hpp")

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

    with ThreadPoolExecutor(max_workers=8) as pool:
        host_objects = [pool.submit(_host_object, name, incremental) for name in HOST_SOURCES]     # the longest compilations first
        objects = list(pool.map(compile_one, SOURCES))
        host_objects = [job.result() for job in host_objects]
    link = [compiler, f"--offload-arch={ARCH}", "-shared", "-fPIC", f"-Wl,-soname,{LIBRARY.name}", *map(str, objects), "-o", str(LIBRARY)]
    _run(link, "linking the library")
    _run([os.environ.get("CXX", "g++"), *map(str, host_objects), "-o", str(HOST_LIBRARY), *_host_flags()[1]], "linking the native host path")
    return LIBRARY


if __name__ == "__main__":
    print(build(incremental="--incremental" in sys.argv))
