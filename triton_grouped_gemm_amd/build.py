"""Compile csrc/*.hip for gfx950 into libtgg_amd.so next to this file, and csrc/host.cpp (the native call path of the
Python entry points, an extension module over torch's C++ API) into _host.so beside it.

``python -m triton_grouped_gemm_amd.build`` (or ``build_library()``) runs hipcc once per
translation unit in parallel and links the objects.  hipcc cross-compiles, so no
GPU is needed to build.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

from .assembly_checks import findings

PKG_DIR = Path(__file__).resolve().parent
CSRC = PKG_DIR / "csrc"
LIB_PATH = PKG_DIR / "libtgg_amd.so"
HOST_PATH = PKG_DIR / "_host.so"
ARCH = "gfx950"
# packed fp32 VALU forms are switched off for every HIP translation unit
HIPCC_FLAGS = ["--offload-arch=" + ARCH, "-O3", "-std=c++17", "-fPIC", "-Xclang", "-target-feature", "-Xclang",
               "-packed-fp32-ops", "-Wno-unused-command-line-argument"]


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(exe).exists():
        raise RuntimeError("hipcc not found; ROCm toolchain is required to build libtgg_amd.so")
    return exe


def _run(cmd):
    proc = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in proc.stderr.splitlines() if noise not in l)
    if proc.returncode != 0:
        raise RuntimeError("command failed: " + " ".join(map(str, cmd)) + "\n" + err)
    return err


def _compile_host(obj: Path):
    """csrc/host.cpp against torch's headers, by the host compiler."""
    from torch.utils.cpp_extension import include_paths
    includes = [*include_paths("cuda"), sysconfig.get_paths()["include"]]
    _run([shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
          *(f"-I{d}" for d in includes), "-c", str(CSRC / "host.cpp"), "-o", str(obj)])


def _link_host(obj: Path):
    """_host.so: finds libtgg_amd.so beside itself and torch's libraries where the running process has loaded them."""
    from torch.utils.cpp_extension import library_paths
    tmp = HOST_PATH.with_suffix(".so.tmp")
    _run([shutil.which("g++") or "g++", "-shared", "-o", str(tmp), str(obj), *(f"-L{d}" for d in library_paths("cuda")),
          "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip", f"-L{PKG_DIR}", f"-l:{LIB_PATH.name}", "-Wl,-rpath,$ORIGIN"])
    os.replace(tmp, HOST_PATH)


def build_library(verbose: bool = False, jobs: int | None = None) -> Path:
    hipcc = _hipcc()
    obj_dir = PKG_DIR / "build"
    obj_dir.mkdir(exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    objs = [obj_dir / (s.stem + ".o") for s in sources]
    jobs = jobs or min(len(sources), int(os.environ.get("MAX_JOBS", "8")))

    def compile_one(pair):
        src, obj = pair
        # -save-temps=obj leaves the intermediate files next to the object; only the device assembly is kept
        # (build/<stem>.gfx950.s) and looked over for what the compiler cannot check around the inline assembly.
        msg = _run([hipcc, *HIPCC_FLAGS, "-save-temps=obj", "-c", str(src), "-o", str(obj)])
        for tmp in obj_dir.glob(src.stem + "*"):
            if tmp == obj:
                continue
            if tmp.name == f"{src.stem}-hip-amdgcn-amd-amdhsa-{ARCH}.s":
                os.replace(tmp, obj_dir / f"{src.stem}.{ARCH}.s")
            elif tmp.suffix != ".s" or "-" in tmp.name:
                tmp.unlink()
        wrong = findings(src.stem, (obj_dir / f"{src.stem}.{ARCH}.s").read_text())
        if wrong:
            raise RuntimeError("the device assembly breaks a rule of assembly_checks.py:\n" + "\n".join(wrong))
        if verbose and msg.strip():
            print(msg, file=sys.stderr)

    host_obj = obj_dir / "host.o"
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        host = pool.submit(_compile_host, host_obj)
        list(pool.map(compile_one, zip(sources, objs)))
        host.result()
    tmp = LIB_PATH.with_suffix(".so.tmp")
    _run([hipcc, "--offload-arch=" + ARCH, "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)])
    os.replace(tmp, LIB_PATH)
    _link_host(host_obj)
    return LIB_PATH


if __name__ == "__main__":
    print(build_library(verbose=True))
