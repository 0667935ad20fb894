"""Build libmoc_hip.so (gfx950) from csrc/*.hip with hipcc, and the host module
that calls it, _moc_host.so, from csrc/moc_host.cpp with g++ against torch.

    python mixture-of-convolutions_amd/build_lib.py [--jobs N]

Objects go to csrc/_build/, both libraries next to the Python package
(moc/), where moc/_lib.py loads them.  Every call recompiles.  libmoc_hip.so
needs hipcc only and is linked first; without torch, Python's headers or g++ the
host module is left out (the Python functions of moc/ then do its calls).
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import importlib.util
import os
import shutil
import subprocess
import sys
import sysconfig
from pathlib import Path

PKG_ROOT = Path(__file__).resolve().parent
CSRC = PKG_ROOT / "csrc"
BUILD = CSRC / "_build"
LIB = PKG_ROOT / "moc" / "libmoc_hip.so"
HOST = PKG_ROOT / "moc" / "_moc_host.so"
ARCH = "gfx950"

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

COMMON_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fno-gpu-rdc",
    # packed FP32 VALU ops are kept out of the device code (some forms of them have
    # given wrong results)
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # MFMA results in VGPRs: the kernels read every result on VALU right away,
    # and AGPR results would cost a v_accvgpr_read per value
    "-mllvm", "-amdgpu-mfma-vgpr-form",
    "-Wall",
    "-Wno-unused-function",
    "-Wno-unused-command-line-argument",
]


def _compile(src: Path, extra: tuple[str, ...] = (), build_dir: Path = BUILD) -> Path:
    obj = build_dir / (src.stem + ".o")
    cmd = [HIPCC, *COMMON_FLAGS, *extra, "-c", str(src), "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    msgs = [ln for ln in (res.stdout + res.stderr).splitlines()
            if "packed-fp32-ops' is not a recognized feature" not in ln]
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n" + "\n".join(msgs))
    if msgs:
        print("\n".join(msgs), file=sys.stderr)
    return obj


CXX = os.environ.get("CXX", "g++")


def host_needs() -> str | None:
    """What the host module's build lacks here, or None."""
    if shutil.which(CXX) is None:
        return f"a C++ compiler ({CXX})"
    torch = importlib.util.find_spec("torch")
    if torch is None or not (Path(torch.origin).parent / "lib" / "libc10_hip.so").exists():
        return "torch for ROCm"
    if not (Path(sysconfig.get_path("include")) / "Python.h").exists():
        return "Python's headers"
    return None


def _compile_host(build_dir: Path) -> Path:
    import torch
    inc = Path(torch.__file__).parent / "include"
    obj = build_dir / "moc_host.o"
    cmd = [CXX, "-O2", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__=1",
           "-DUSE_ROCM=1", "-DTORCH_EXTENSION_NAME=_moc_host",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           f"-I{inc}", f"-I{inc / 'torch/csrc/api/include'}", f"-I{Path(HIPCC).parents[1] / 'include'}",
           f"-I{sysconfig.get_path('include')}", "-c", str(CSRC / "moc_host.cpp"), "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("moc_host.cpp failed:\n" + res.stdout + res.stderr)
    return obj


def _link_host(obj: Path) -> None:
    import torch
    lib = Path(torch.__file__).parent / "lib"
    tmp = HOST.with_suffix(".so.tmp")
    cmd = [CXX, "-shared", "-o", str(tmp), str(obj), f"-L{lib}", "-ltorch_python",
           "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip", f"-L{LIB.parent}",
           f"-l:{LIB.name}", "-Wl,-rpath,$ORIGIN"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("link of the host module failed:\n" + res.stdout + res.stderr)
    os.replace(tmp, HOST)


def build(jobs: int | None = None, verbose: bool = True, defines: tuple[str, ...] = (),
          out: Path = LIB) -> Path:
    """Compile csrc/*.hip and link ``out``; ``defines`` are extra -D flags."""
    if shutil.which(HIPCC) is None and not Path(HIPCC).exists():
        raise RuntimeError(f"hipcc not found at {HIPCC}")
    build_dir = BUILD if not defines else BUILD / ("_".join(defines).replace("=", "-"))
    build_dir.mkdir(parents=True, exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    jobs = jobs or min(len(sources), max(1, (os.cpu_count() or 4)))
    extra = tuple(f"-D{d}" for d in defines)
    LIB_OUT = Path(out)
    lacks = host_needs() if LIB_OUT == LIB else "not asked for"
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        host = ex.submit(_compile_host, build_dir) if lacks is None else None
        objs = list(ex.map(lambda src: _compile(src, extra, build_dir), sources))
    tmp = LIB_OUT.with_suffix(".so.tmp")
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("link failed:\n" + res.stdout + res.stderr)
    os.replace(tmp, LIB_OUT)
    if LIB_OUT == LIB:
        HOST.unlink(missing_ok=True)  # (one of another build of the library)
        if host is not None:
            _link_host(host.result())
        else:
            print(f"host module not built: needs {lacks}", file=sys.stderr)
    if verbose:
        print(f"built {LIB_OUT} from {len(sources)} sources")
    return LIB_OUT


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=None)
    ap.add_argument("-D", dest="defines", action="append", default=[],
                    help="extra preprocessor define, e.g. -D MOC_BWD_MIN_WAVES=2")
    ap.add_argument("--out", default=str(LIB))
    a = ap.parse_args()
    build(a.jobs, defines=tuple(a.defines), out=Path(a.out))
