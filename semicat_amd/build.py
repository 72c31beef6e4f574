"""Builds libsjvp.so (the gfx950 attention-JVP kernels + C ABI) in-tree with hipcc.

The kernels are instantiated in several translation units (one per kernel family and element type)
that are compiled in parallel and linked into one shared library.  Beside it goes a small CPython extension,
the host side of the entry points (csrc/sjvp_host.cpp)."""
from __future__ import annotations

import hashlib
import os
import re
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(PKG_DIR, "csrc")
OBJ_DIR = os.path.join(PKG_DIR, "build")
LIB_PATH = os.path.join(PKG_DIR, "libsjvp.so")
# (source, element types it is compiled for: the unit instantiates its kernels for -DSJVP_T=<type>)
UNITS = [(name, ("Bf16", "Fp16") if name.startswith("sjvp_tu_") else (None,))
         for name in sorted(os.listdir(CSRC)) if name.endswith(".hip")]
SOURCES = [os.path.join(CSRC, name) for name, _ in UNITS]
# The host side of the entry points: a CPython extension against torch's headers, no device code.
HOST_SOURCE = os.path.join(CSRC, "sjvp_host.cpp")
HOST_PATH = os.path.join(PKG_DIR, "_sjvp_host.so")
ABI_HEADER = os.path.join(os.path.dirname(PKG_DIR), "include", "sjvp.h")
HEADERS = sorted(os.path.join(CSRC, n) for n in os.listdir(CSRC) if n.endswith(".hpp")) + [ABI_HEADER]

HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++20", "-fPIC",
    # keep the compiler from forming packed-fp32 instructions
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]
# Flags of single units.  The row-owned and column-owned backward kernels gain 1 to 4 % from the
# scheduler that orders for instruction-level parallelism (measured on the MI355X at head dimensions 64 and
# 128); the single-launch backward loses 2 % with it, the forward is unchanged on aligned rows and loses up
# to 20 % on staged ones, so they keep the default.
_ILP = ["-mllvm", "-amdgpu-sched-strategy=max-ilp"]
UNIT_FLAGS = {name: _ILP for name in ("sjvp_tu_pair16.hip", "sjvp_tu_pair_staged16.hip", "sjvp_f32io_pair.hip")}
# Accumulators among the vector registers.  Forward + backward without tangents, without / with it: B=4 H=16 L=2048 D=64 1756 / 1650 us, B=8
# H=12 L=500 D=96 448 / 435, twelve shapes 1.035; with tangents 1.004.  The same registers are spilled either way.
UNIT_FLAGS["sjvp_f32x3.hip"] = ["-mllvm", "-amdgpu-mfma-vgpr-form=1"]


def hipcc_path() -> str:
    for cand in (shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (expected on PATH or at /opt/rocm/bin/hipcc)")


# Flags of the host extension (g++; the include and library folders of torch, ROCm and Python come on top).
HOST_FLAGS = ["-O2", "-std=c++20", "-fPIC", "-shared", "-w", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1"]
HOST_LIBS = ["-ltorch_python", "-ltorch_hip", "-ltorch_cpu", "-lc10_hip", "-lc10"]


def _hash(what: str, paths) -> str:
    h = hashlib.sha256(what.encode())
    for path in paths:
        h.update(os.path.basename(path).encode())
        with open(path, "rb") as f:
            h.update(f.read())
    return h.hexdigest()[:16]


def source_id() -> str:
    """Identifier of the sources the library is built from: a hash of their contents and the flags."""
    return _hash(" ".join(HIPCC_FLAGS) + repr(sorted(UNIT_FLAGS.items())), SOURCES + HEADERS)


def host_id() -> str:
    """Identifier of what the host extension is built from: its source, the C ABI it calls, the flags, and the torch and
    interpreter whose headers it is compiled against (inlined accessors read torch's object layouts)."""
    import torch
    against = (torch.__version__, torch.version.hip, torch.compiled_with_cxx11_abi(), sysconfig.get_config_var("SOABI"))
    return _hash(repr((HOST_FLAGS, HOST_LIBS, against)), [HOST_SOURCE, ABI_HEADER])


def built_id(path: str = LIB_PATH) -> str | None:
    """The source identifier embedded in a built library (read from the file, nothing is loaded)."""
    try:
        with open(path, "rb") as f:
            m = re.search(rb"SJVP_BUILD_ID=([0-9a-f]{16})", f.read())
    except OSError:
        return None
    return m.group(1).decode() if m else None


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), file=sys.stderr)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("the compiler failed:\n" + " ".join(cmd) + "\n" + res.stdout + res.stderr)


def host_command() -> list[str]:
    """The command that builds the host extension (host code only: g++)."""
    import torch
    root = os.path.dirname(torch.__file__)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    return [shutil.which("g++") or "c++", *HOST_FLAGS, f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}",
            f'-DSJVP_BUILD_ID="SJVP_BUILD_ID={host_id()}"', "-I" + sysconfig.get_paths()["include"], "-I" + os.path.join(root, "include"),
            "-I" + os.path.join(root, "include", "torch", "csrc", "api", "include"), "-I" + os.path.join(rocm, "include"),
            HOST_SOURCE, "-o", HOST_PATH + ".tmp", "-L" + os.path.join(root, "lib"), *HOST_LIBS]


def build_host(verbose: bool = False) -> str:
    """Compile the host extension; returns its path."""
    _run(host_command(), verbose)
    os.replace(HOST_PATH + ".tmp", HOST_PATH)
    return HOST_PATH


def build_library(verbose: bool = False, jobs: int | None = None) -> str:
    """Compile every translation unit of the C library unconditionally and link; needs nothing but hipcc."""
    hipcc = hipcc_path()
    os.makedirs(OBJ_DIR, exist_ok=True)
    cmds, objs = [], []
    build_id = f'-DSJVP_BUILD_ID="SJVP_BUILD_ID={source_id()}"'
    for name, types in UNITS:
        for t in types:
            obj = os.path.join(OBJ_DIR, name[:-4] + (f"_{t}" if t else "") + ".o")
            define = [f"-DSJVP_T={t}"] if t else ([build_id] if name == "sjvp_api.hip" else [])
            cmds.append([hipcc, *HIPCC_FLAGS, *UNIT_FLAGS.get(name, []), *define, "-c", os.path.join(CSRC, name),
                         "-o", obj])
            objs.append(obj)
    jobs = jobs or min(len(cmds), os.cpu_count() or 4, 16)
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        list(pool.map(lambda c: _run(c, verbose), cmds))
    _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB_PATH + ".tmp", *objs], verbose)
    os.replace(LIB_PATH + ".tmp", LIB_PATH)
    return LIB_PATH


def build(verbose: bool = False, jobs: int | None = None) -> str:
    """Compile everything unconditionally; returns the path of the library.  Where the host extension fails to build, the
    library is there all the same when the error comes."""
    with ThreadPoolExecutor(max_workers=1) as beside:
        host = beside.submit(build_host, verbose)
        path = build_library(verbose, jobs)
        host.result()
    return path


def library_is_stale() -> bool:
    """True when no library is built or one from other sources than the ones in the tree (compared by content, so copying
    or checking out the tree does not matter)."""
    return built_id(LIB_PATH) != source_id()


def host_is_stale() -> bool:
    """The same of the host extension, which is also stale beside another torch or interpreter than its own."""
    return built_id(HOST_PATH) != host_id()


def is_stale() -> bool:
    """True when the library or the host extension is."""
    return library_is_stale() or host_is_stale()


if __name__ == "__main__":
    print(build_library(verbose=True))
    print(build_host(verbose=True))
