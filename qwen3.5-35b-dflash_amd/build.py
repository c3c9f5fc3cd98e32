"""Build recipe for ``libdflash_hip.so`` (hand-written HIP for gfx950 only) and ``dflash_host.so`` (the native form
of ops.py's plain calls: C++ over torch's headers, no device code).

``python build.py`` from this directory, or ``build()`` from Python.  Each
translation unit is compiled in parallel with hipcc, then linked into one
shared library next to this file; the library is replaced atomically.
``python build.py --timeline`` (``build(timeline=True)``) builds the profiling
variant ``libdflash_hip_timeline.so`` instead: the same kernels with phase
timestamps (``-DDFLASH_TIMELINE``), loaded only by ``timeline.py``.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
import tempfile
from pathlib import Path

PACKAGE_DIR = Path(__file__).resolve().parent
LIBRARY = PACKAGE_DIR / "libdflash_hip.so"
TIMELINE_LIBRARY = PACKAGE_DIR / "libdflash_hip_timeline.so"
SOURCES = ("csrc/api.hip", "csrc/route.hip", "csrc/w4_gemm.hip", "csrc/w4_stream.hip",
           "csrc/w4_tile.hip", "csrc/w4_verify.hip", "csrc/w4_small.hip", "csrc/w4_linear.hip",
           "csrc/repack.hip", "csrc/gdn.hip", "csrc/attention.hip")
HOST_SOURCE = "csrc/host.cpp"
HOST_LIBRARY = PACKAGE_DIR / "dflash_host.so"
ARCH = "gfx950"
FLAGS = (
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    # keep the compiler from forming packed-fp32 VALU ops (v_pk_*_f32)
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
)


def _hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(path).exists():
        raise RuntimeError("hipcc not found; a ROCm toolchain is required to build libdflash_hip.so")
    return path


def _host_command(output: Path) -> list:
    import torch
    root = Path(torch.__file__).resolve().parent
    include = (root / "include", root / "include/torch/csrc/api/include", sysconfig.get_paths()["include"],
               "/opt/rocm/include")
    return [shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-DUSE_ROCM=1", "-D__HIP_PLATFORM_AMD__=1",
            f'-DDFLASH_TORCH="{torch.__version__}"',
            *(f"-I{i}" for i in include), str(PACKAGE_DIR / HOST_SOURCE), "-o", str(output), f"-L{root / 'lib'}",
            "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip"]


def _start(cmd: list) -> tuple:
    return cmd, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)


def _start_host(output: Path):
    """The compile of the host library, or None where g++ or torch is missing."""
    try:
        return _start(_host_command(output))
    except (ImportError, OSError) as error:
        print(f"{HOST_LIBRARY.name} is not built: {error}", file=sys.stderr)
        return None


def _finish_host(job) -> bool:
    """Whether the host library was compiled.  Without it every call takes its Python form."""
    if job is None:
        return False
    out, _ = job[1].communicate()
    if job[1].returncode:
        print(f"{HOST_LIBRARY.name} is not built: {' '.join(job[0])}\n{out}", file=sys.stderr)
    return job[1].returncode == 0


def _install(built: Path, final: Path) -> None:
    tmp_target = final.with_suffix(".so.tmp")
    shutil.copyfile(built, tmp_target)
    os.replace(tmp_target, final)


def build(verbose: bool = False, timeline: bool = False) -> Path:
    hipcc = _hipcc()
    target = TIMELINE_LIBRARY if timeline else LIBRARY
    flags = (*FLAGS, "-DDFLASH_TIMELINE") if timeline else FLAGS
    with tempfile.TemporaryDirectory(prefix="dflash_build_") as tmp:
        objects, procs = [], []
        for src in SOURCES:
            obj = Path(tmp) / (Path(src).stem + ".o")
            cmd = [hipcc, *flags, "-c", str(PACKAGE_DIR / src), "-o", str(obj)]
            objects.append(obj)
            procs.append(_start(cmd))
        host = Path(tmp) / HOST_LIBRARY.name
        job = None if timeline else _start_host(host)
        for cmd, proc in procs:
            out, _ = proc.communicate()
            if proc.returncode:
                raise RuntimeError(f"compiler failed ({proc.returncode}): {' '.join(cmd)}\n{out}")
            if verbose and out.strip():
                print(out)
        staged = Path(tmp) / target.name
        link = [hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objects), "-o", str(staged)]
        proc = subprocess.run(link, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
        if proc.returncode:
            raise RuntimeError(f"link failed: {' '.join(link)}\n{proc.stdout}")
        _install(staged, target)
        if not timeline:
            if _finish_host(job):
                _install(host, HOST_LIBRARY)
            else:
                HOST_LIBRARY.unlink(missing_ok=True)  # not one of other sources or another torch
    return target


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv, timeline="--timeline" in sys.argv))
