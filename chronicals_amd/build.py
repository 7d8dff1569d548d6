"""Build libchronicals_cce.so (HIP, gfx950) and the torch operators over it in-tree.

The library is compiled with hipcc from ``chronicals_amd/csrc/cce_kernels.hip``
into ``chronicals_amd/lib/libchronicals_cce.so``; the package loads it from
there with ctypes.  The torch operators (``csrc/torch_ops.cpp``, host code only)
are compiled against the installed torch into
``lib/libchronicals_torch-<hash>-<torch version>.so``, where the hash covers
their source and the header: a build of anything else has another name and is
never loaded.  Building always recompiles both, the HIP library first: it needs
neither torch nor a host compiler, and stays usable from C where the operators
cannot be built.
"""
from __future__ import annotations

import hashlib
import importlib.util
import os
import shutil
import subprocess
import sys
import sysconfig

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
REPO_DIR = os.path.dirname(PKG_DIR)
SRC = os.path.join(PKG_DIR, "csrc", "cce_kernels.hip")
HEADER = os.path.join(REPO_DIR, "include", "chronicals_cce.h")
TORCH_SRC = os.path.join(PKG_DIR, "csrc", "torch_ops.cpp")
LIB_DIR = os.path.join(PKG_DIR, "lib")
LIB_NAME = "libchronicals_cce.so"
LIB_PATH = os.path.join(LIB_DIR, LIB_NAME)
# per-kernel register / LDS / spill report of the last build (compiler remarks)
RESOURCES_PATH = os.path.join(LIB_DIR, "libchronicals_cce.resources.txt")
ARCH = "gfx950"


def hipcc_path() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found: the HIP toolchain (ROCm) is required to build chronicals_amd")


def source_hash(paths=(SRC, HEADER)) -> str:
    """SHA-256 (hex) over the files the library is compiled from, in order.
    The build compiles it into the library (cce_source_hash()), so the loader
    can tell a library built from other sources."""
    h = hashlib.sha256()
    for p in paths:
        with open(p, "rb") as f:
            data = f.read()
        h.update(os.path.basename(p).encode() + b"\0" + str(len(data)).encode() + b"\0" + data)
    return h.hexdigest()


def compile_command(out_path: str, src_hash: str = None) -> list:
    return [
        hipcc_path(),
        f"--offload-arch={ARCH}",
        "-O3",
        "-std=c++17",
        "-fPIC",
        "-shared",
        # packed fp32 VALU ops stay off (the compiler may not form them)
        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
        "-I", os.path.join(REPO_DIR, "include"),
        # bare hex digits (the source stringifies them): no shell quoting involved
        f"-DCCE_SOURCE_HASH={src_hash or source_hash()}",
        # per-kernel resource usage (VGPRs, spills, LDS) as compiler remarks
        "-Rpass-analysis=kernel-resource-usage",
        "-o", out_path,
        SRC,
    ]


def torch_lib_path() -> str:
    """Where the torch operators of this tree and this torch are built.  Without
    the sources (an installed tree): the one build for this torch."""
    import torch

    tail = f"-{torch.__version__}.so"
    if not (os.path.exists(TORCH_SRC) and os.path.exists(HEADER)):
        built = [n for n in (os.listdir(LIB_DIR) if os.path.isdir(LIB_DIR) else ())
                 if n.startswith("libchronicals_torch-") and n.endswith(tail)]
        return os.path.join(LIB_DIR, built[0] if len(built) == 1 else f"libchronicals_torch-*{tail}")
    return os.path.join(LIB_DIR, f"libchronicals_torch-{source_hash((TORCH_SRC, HEADER))[:16]}{tail}")


def torch_compile_command(out_path: str) -> list:
    import torch

    base = os.path.dirname(torch.__file__)
    inc, lib = os.path.join(base, "include"), os.path.join(base, "lib")
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(hipcc_path())))
    return [
        shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared",
        # what torch's ROCm headers ask of their users
        "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
        f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
        "-isystem", inc, "-isystem", os.path.join(inc, "torch", "csrc", "api", "include"),
        "-isystem", os.path.join(rocm, "include"), "-isystem", sysconfig.get_paths()["include"],
        TORCH_SRC, "-o", out_path,
        "-L", lib, "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch", "-ltorch_python", f"-Wl,-rpath,{lib}",
    ]


def build_torch(verbose: bool = False) -> str:
    """Compile the torch operators; returns the path of the built .so and removes builds of other sources."""
    os.makedirs(LIB_DIR, exist_ok=True)
    path = torch_lib_path()
    tmp = path + f".tmp{os.getpid()}"
    cmd = torch_compile_command(tmp)
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        sys.stderr.write(proc.stdout + proc.stderr)
        raise RuntimeError(f"g++ failed with exit code {proc.returncode}")
    os.replace(tmp, path)
    for name in os.listdir(LIB_DIR):
        if name.startswith("libchronicals_torch-") and name.endswith(".so") and name != os.path.basename(path):
            os.remove(os.path.join(LIB_DIR, name))
    return path


def parse_resources(text: str) -> dict:
    """{kernel symbol: {field: int}} from kernel-resource-usage remarks."""
    out, cur = {}, None
    for line in text.splitlines():
        if "remark:" not in line:
            continue
        body = line.split("remark:", 1)[1].strip()
        body = body.split(" [-Rpass", 1)[0]
        if body.startswith("Function Name:"):
            cur = out.setdefault(body.split(":", 1)[1].strip(), {})
        elif cur is not None and ":" in body:
            key, val = body.split(":", 1)
            try:
                cur[key.strip()] = int(val.strip().split()[0])
            except ValueError:
                pass
    return out


def build(verbose: bool = False) -> str:
    """Compile the HIP library and, where torch is installed, its operators; returns the path of the HIP library."""
    build_hip(verbose)
    if importlib.util.find_spec("torch") is None:
        sys.stderr.write("torch is not installed: its operators are not built\n")
    else:
        build_torch(verbose)
    return LIB_PATH


def build_hip(verbose: bool = False) -> None:
    """Compile the HIP library."""
    os.makedirs(LIB_DIR, exist_ok=True)
    tmp = LIB_PATH + f".tmp{os.getpid()}"
    cmd = compile_command(tmp, source_hash())
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        sys.stderr.write(proc.stdout + proc.stderr)
        raise RuntimeError(f"hipcc failed with exit code {proc.returncode}")
    os.replace(tmp, LIB_PATH)
    res = parse_resources(proc.stdout + proc.stderr)
    with open(RESOURCES_PATH, "w") as f:
        for name in sorted(res):
            f.write(name + " " + " ".join(f"{k.replace(' ', '_')}={v}" for k, v in sorted(res[name].items())) + "\n")
    spills = {n: r.get("VGPRs Spill", 0) for n, r in res.items() if r.get("VGPRs Spill", 0)}
    if spills:
        sys.stderr.write(f"warning: kernels spill VGPRs to scratch: {spills}\n")


if __name__ == "__main__":
    print(build(verbose=True))
