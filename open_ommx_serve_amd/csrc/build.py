"""Build the native code in-tree for gfx950.

    python -m open_ommx_serve_amd.csrc.build

Each .hip file is compiled to an object and the objects are linked into ``libommx_hip.so`` next
to the sources.  The store kernels are compiled with floating-point contraction off: their
arithmetic has to round exactly where the reference packer rounds.  ``ommx_host.cpp``, the
native half of the Python launchers, becomes the extension module ``_ommx_host`` beside it.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(HERE, "libommx_hip.so")
HOST_MODULE = os.path.join(HERE, "_ommx_host" + sysconfig.get_config_var("EXT_SUFFIX"))
ARCH = "gfx950"
SOURCES = {
    "ommx_store.hip": ["-ffp-contract=off"],
    "ommx_store_long.hip": ["-ffp-contract=off"],
    "ommx_store_generic.hip": ["-ffp-contract=off"],
    "ommx_decode_ref.hip": [],
    "ommx_decode.hip": [],
    "ommx_decode_gqa4.hip": [],
    "ommx_decode_gqa4_tail.hip": [],
    "ommx_decode_team.hip": [],
    "ommx_decode_fp32.hip": [],
    "ommx_combine.hip": [],
    "ommx_ring.hip": [],
    "ommx_merge.hip": [],
    "ommx_index.hip": [],
    "ommx_prefill.hip": [],
    "ommx_capi.hip": [],
}
COMMON = ["-O3", "-fPIC", "-std=c++17", f"--offload-arch={ARCH}",
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
          "-Wno-unused-command-line-argument"]


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; libommx_hip.so cannot be built")
    return exe


def _run(cmd, what: str):
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{what} failed:\n{r.stdout}\n{r.stderr}")
    noise = [ln for ln in r.stderr.splitlines()
             if ln.strip() and "packed-fp32-ops" not in ln and "not a recognized feature" not in ln]
    if noise:
        print("\n".join(noise), file=sys.stderr)


def _compile(src: str, extra) -> str:
    obj = os.path.join(HERE, src.replace(".hip", ".o"))
    _run([_hipcc(), *COMMON, *extra, "-c", os.path.join(HERE, src), "-o", obj], f"hipcc on {src}")
    return obj


def _compile_host() -> str:
    """Host C++ only (no kernel in it; HIP's own headers ask g++ for the platform macro); ``-isystem``: warnings of torch's own headers are not ours."""
    from torch.utils.cpp_extension import include_paths
    obj = os.path.join(HERE, "ommx_host.o")
    inc = [f"-isystem{p}" for p in (*include_paths("cuda"), sysconfig.get_paths()["include"])]
    _run(["g++", "-O2", "-fPIC", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", *inc,
          "-c", os.path.join(HERE, "ommx_host.cpp"), "-o", obj], "g++ on ommx_host.cpp")
    return obj


def build(verbose: bool = True) -> str:
    from torch.utils.cpp_extension import library_paths
    with ThreadPoolExecutor(max_workers=8) as ex:
        host = ex.submit(_compile_host)
        objs = list(ex.map(lambda kv: _compile(*kv), SOURCES.items()))
        host_obj = host.result()
    _run([_hipcc(), "-shared", "-fPIC", f"--offload-arch={ARCH}", *objs, "-o", LIB], "link of libommx_hip.so")
    torch_libs = [p for p in library_paths() if os.path.exists(os.path.join(p, "libtorch_python.so"))]
    _run(["g++", "-shared", host_obj, "-o", HOST_MODULE, f"-L{HERE}", "-l:libommx_hip.so", "-Wl,-rpath,$ORIGIN",
          *(f"-L{p}" for p in torch_libs), "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip",
          "-lamdhip64"], "link of _ommx_host")
    if verbose:
        for path in (LIB, HOST_MODULE):
            print(f"built {path} ({os.path.getsize(path)} bytes)")
    return LIB


if __name__ == "__main__":
    build()
