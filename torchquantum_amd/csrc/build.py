"""Build ``libtqsv.so`` (all HIP kernels + the C ABI) for gfx950 with hipcc, and
``_tqhost.so`` (the host path of a call, a CPython extension) with g++.

Usage: ``python -m torchquantum_amd.csrc.build`` or ``build()`` from Python.
Both are written in-tree next to this package (``torchquantum_amd/``) so that they
travel with the source tree.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
import tempfile
from pathlib import Path

HERE = Path(__file__).resolve().parent
PKG = HERE.parent
LIB = PKG / "libtqsv.so"
HOST = PKG / "_tqhost.so"
HOST_SOURCE = "tqsv_host.cpp"

SOURCES = [
    "tqsv_gates.hip",
    "tqsv_stage.hip",
    "tqsv_expval.hip",
    "tqsv_adjoint.hip",
    "tqsv_devgates.hip",
    "tqsv_mlp.hip",
    "tqsv_sample.hip",
    "tqsv_jit.hip",
]

ARCH = os.environ.get("TQSV_ARCH", "gfx950")

FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fvisibility=hidden",
    "-munsafe-fp-atomics",
    # no packed-FP32 (v_pk_*_f32) instructions anywhere
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def hipcc() -> str:
    for c in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if c and Path(c).exists():
            return c
    raise RuntimeError("hipcc not found (ROCm is required to build libtqsv.so)")


def host_command(out: Path) -> list:
    """g++ command that builds the host extension against the installed torch and this Python."""
    import sysconfig
    import torch
    inc = Path(torch.__file__).parent / "include"
    cxx = os.environ.get("CXX") or shutil.which("g++") or "g++"
    return [cxx, "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-w",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}",
            "-I", str(inc), "-I", str(inc / "torch/csrc/api/include"), "-I", sysconfig.get_paths()["include"],
            str(HERE / HOST_SOURCE), "-o", str(out), "-L", str(Path(torch.__file__).parent / "lib"),
            "-ltorch_python", "-ltorch_cpu", "-lc10"]


def build(verbose: bool = False, jobs: int = 6) -> Path:
    """Compile every source to an object, link the shared library and build the host extension."""
    cc = hipcc()
    srcs = [HERE / s for s in SOURCES]
    missing = [str(p) for p in srcs + [HERE / HOST_SOURCE] if not p.exists()]
    if missing:
        raise RuntimeError(f"libtqsv.so sources missing: {missing}")
    tmp = Path(tempfile.mkdtemp(prefix="tqsv_build_"))
    try:
        tmp_host = tmp / HOST.name
        host = subprocess.Popen(host_command(tmp_host), stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
        procs = []
        objs = []
        for src in srcs:
            obj = tmp / (src.stem + ".o")
            cmd = [cc, *FLAGS, "-I", str(HERE), "-c", str(src), "-o", str(obj)]
            if verbose:
                print(" ".join(cmd), flush=True)
            procs.append((src, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)))
            objs.append(obj)
            while sum(p.poll() is None for _, p in procs) >= jobs:
                procs[[p.poll() is None for _, p in procs].index(True)][1].wait()
        failed = []
        for src, p in procs:
            out = p.communicate()[0].decode(errors="replace")
            out = "\n".join(l for l in out.splitlines() if "packed-fp32-ops" not in l)
            if p.returncode != 0:
                failed.append(f"--- {src.name}\n{out}")
            elif verbose and out.strip():
                print(out)
        out = host.communicate()[0].decode(errors="replace")
        if host.returncode != 0:
            failed.append(f"--- {HOST_SOURCE}\n{out}")
        if failed:
            raise RuntimeError("compile failed:\n" + "\n".join(failed))
        tmp_lib = tmp / "libtqsv.so"
        cmd = [cc, f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objs), "-o", str(tmp_lib),
               "-lhiprtc"]
        r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
        if r.returncode != 0:
            raise RuntimeError("link failed:\n" + r.stdout.decode(errors="replace"))
        shutil.move(str(tmp_lib), str(LIB))
        shutil.move(str(tmp_host), str(HOST))
        return LIB
    finally:
        shutil.rmtree(tmp, ignore_errors=True)


if __name__ == "__main__":
    p = build(verbose="-v" in sys.argv)
    print(p)
