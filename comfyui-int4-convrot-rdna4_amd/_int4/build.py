"""Ahead-of-time build of the gfx950 kernel library (replaces the reference's
JIT ``_int4/build.py``, which compiled for whatever arch the GPU reported).

``build()`` runs hipcc for gfx950 only: every source is compiled to an object
in parallel (``_build/`` next to this file), then the objects are linked into
``libconvrot_gfx950.so`` next to this file, and the host module ``_host.so``
(csrc/host.cpp) against it.  Both are loaded by
``native.py``; nothing builds at import or at first use.
"""
from __future__ import annotations

import importlib.util
import os
import shutil
import subprocess
import sysconfig
from concurrent.futures import ThreadPoolExecutor

_HERE = os.path.dirname(os.path.abspath(__file__))
_PKG = os.path.dirname(_HERE)
_CSRC = os.path.join(_PKG, "csrc")
SOURCES = ("rotquant.hip", "gemm.hip", "gemm_bf6.hip", "gemm_bf6_direct.hip", "gemm_int.hip", "lora.hip", "dequant.hip", "capi.hip")
HEADERS = ("common.h", "gemm_common.h", "gemm_direct.h", "gemm_int.h", "b6t_layout.h")
ARCH = "gfx950"


def lib_path() -> str:
    return os.path.join(_HERE, "libconvrot_gfx950.so")


def host_path() -> str:
    return os.path.join(_HERE, "_host.so")


def sources() -> list[str]:
    return [os.path.join(_CSRC, s) for s in SOURCES]


def _deps() -> list[str]:
    return sources() + [os.path.join(_CSRC, h) for h in HEADERS + ("host.cpp",)] + [
        os.path.join(os.path.dirname(_PKG), "include", "convrot_mi355x.h")]


def is_stale() -> bool:
    """Whether a source is newer than what was built from it, or the host module
    older than the library it is linked to (a build that ended between the two)."""
    out, host = lib_path(), host_path()
    if not os.path.exists(out) or not os.path.exists(host):
        return True
    t = os.path.getmtime(out)
    return os.path.getmtime(host) < t or any(os.path.getmtime(d) > t for d in _deps() if os.path.exists(d))


def _hipcc() -> str:
    return shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


# Flags of every translation unit.  -ffp-contract=off keeps the epilogue's
# separately rounded products and sums; packed-fp32 VALU forms stay off
# (compiler-generated v_pk_*_f32 disabled).
CFLAGS = ["-O3", "-std=c++17", f"--offload-arch={ARCH}", "-fPIC", "-fvisibility=hidden", "-ffp-contract=off",
          "-fhip-fp32-correctly-rounded-divide-sqrt", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]


def hipcc_cmd(out: str) -> list[str]:
    """One-step command (all sources, one hipcc process); build() uses the
    equivalent compile-then-link steps below."""
    return [_hipcc(), *CFLAGS, "-shared", *sources(), "-o", out]


def _obj_dir() -> str:
    d = os.path.join(_HERE, "_build")
    os.makedirs(d, exist_ok=True)
    return d


def _compile(src: str) -> str:
    obj = os.path.join(_obj_dir(), os.path.basename(src) + ".o")
    tmp = obj + ".tmp"
    cp = subprocess.run([_hipcc(), *CFLAGS, "-c", src, "-o", tmp], capture_output=True, text=True)
    if cp.returncode != 0 or not os.path.exists(tmp):
        raise RuntimeError(f"hipcc failed on {os.path.basename(src)}:\n{cp.stderr}")
    os.replace(tmp, obj)
    return obj


def _torch_dir() -> str:
    return os.path.dirname(importlib.util.find_spec("torch").origin)


def _run(cmd: list[str], out: str, what: str) -> None:
    cp = subprocess.run([*cmd, "-o", out + ".tmp"], capture_output=True, text=True)
    if cp.returncode != 0 or not os.path.exists(out + ".tmp"):
        raise RuntimeError(f"{what} failed:\n{cp.stderr}")
    os.replace(out + ".tmp", out)


def _compile_host() -> str:
    """csrc/host.cpp (host code only) against torch's headers."""
    inc = os.path.join(_torch_dir(), "include")
    rocm = os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(_hipcc()))), "include")
    obj = os.path.join(_obj_dir(), "host.cpp.o")
    _run([_hipcc(), "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-DUSE_ROCM", "-D__HIP_PLATFORM_AMD__",
          "-isystem", inc, "-isystem", os.path.join(inc, "torch", "csrc", "api", "include"),
          "-isystem", sysconfig.get_paths()["include"], "-isystem", rocm, "-x", "c++", "-c",
          os.path.join(_CSRC, "host.cpp")], obj, "hipcc on host.cpp")
    return obj


def _link_host(obj: str, lib: str, out: str) -> None:
    """The CPython module, bound to the kernel library next to it."""
    _run([_hipcc(), "-shared", "-fPIC", "-Wl,--as-needed", obj, "-L" + os.path.join(_torch_dir(), "lib"), "-ltorch_python", "-ltorch_cpu",
          "-lc10", "-lc10_hip", "-L" + os.path.dirname(lib), "-l:" + os.path.basename(lib), "-Wl,-rpath,$ORIGIN"],
         out, "linking the host module")


def build(verbose: bool = False, jobs: int | None = None) -> str:
    srcs = sources()
    if verbose:
        print("building:", " ".join([_hipcc(), *CFLAGS, "-c", "<src>"]), "for", ", ".join(SOURCES))
    n = jobs or min(len(srcs) + 1, max(1, (os.cpu_count() or 4)))
    with ThreadPoolExecutor(max_workers=n) as ex:
        host = ex.submit(_compile_host)
        objs = list(ex.map(_compile, srcs))
    # both linked aside under their names, then moved in place: a build that fails leaves the pair that was there
    lib = os.path.join(_obj_dir(), os.path.basename(lib_path()))
    mod = os.path.join(_obj_dir(), os.path.basename(host_path()))
    _run([_hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs], lib, "hipcc link")
    _link_host(host.result(), lib, mod)
    os.replace(lib, lib_path())
    os.replace(mod, host_path())
    return lib_path()


if __name__ == "__main__":
    print("built:", build(verbose=True))
