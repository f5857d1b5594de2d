"""Build libgdnreplay.so (the HIP kernels + the C-ABI layer) for gfx950.

    python gdnr_build.py [-v]

Objects go to _build/ next to this file; the library is written in-tree
(next to this file) so it travels with the source tree to the GPU host.
The C-ABI validation layer (csrc/gdnr_abi.cpp) is plain C++ compiled by g++;
the kernels (csrc/*.hip) by hipcc. Packed-FP32 VALU instructions
are disabled for all device code. The host extension module _gdnr_host.so
(csrc/gdnr_host.cpp, g++ with torch's headers) is written next to the library.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
CSRC = PKG_DIR / "csrc"
INCLUDE = PKG_DIR.parent / "include"
BUILD_DIR = PKG_DIR / "_build"
LIBRARY = PKG_DIR / "libgdnreplay.so"
HOST_MODULE = PKG_DIR / "_gdnr_host.so"
ARCH = os.environ.get("GDNR_OFFLOAD_ARCH", "gfx950")

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def _rocm() -> Path:
    """The ROCm tree hipcc belongs to (its headers go with its compiler)."""
    tree = Path(HIPCC).resolve().parents[1]
    return tree if (tree / "include/hip/hip_runtime_api.h").exists() else Path(os.environ.get("ROCM_PATH", "/opt/rocm"))


DEVICE_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-result",
]
HOST_FLAGS = ["-O2", "-std=c++17", "-fPIC", "-Wall", "-Wextra"]
ACTS = ("bf16", "f16", "f32")  # activation dtypes, one kernel object each (GDNR_ACT = index)
KERNEL_SOURCES = ("gdnr_kernels", "gdnr_step", "gdnr_decode", "gdnr_ring")  # compiled once per activation dtype
SINGLE_SOURCES = ("gdnr_rmw", "gdnr_formats", "gdnr_status", "gdnr_probe")  # compiled once (dtypes are template arguments)
# per-source device flags: the decode kernel's first 13 argument dwords are
# preloaded into SGPRs at wave launch (gfx950 kernarg preload), and its
# wave-uniform branches (workgroup role, replay or flush) are left as scalar
# branches rather than structurised into a chain in which one arm's values
# stay live across the other; the ring kernel likewise
PRELOAD_UNIFORM = ["-mllvm", "-amdgpu-kernarg-preload-count=13", "-mllvm", "-structurizecfg-skip-uniform-regions=true"]
SOURCE_FLAGS = {"gdnr_decode": PRELOAD_UNIFORM, "gdnr_ring": PRELOAD_UNIFORM}


def _run(cmd: list[str], verbose: bool) -> None:
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    stderr = "\n".join(line for line in proc.stderr.splitlines() if noise not in line)
    if proc.returncode != 0:
        raise RuntimeError(f"build step failed ({proc.returncode}): {' '.join(cmd)}\n{stderr}")
    if verbose and stderr.strip():
        print(stderr, file=sys.stderr)


def _host_module_job(out: Path) -> list[str]:
    import torch

    root = Path(torch.__file__).resolve().parent
    return ["g++", *HOST_FLAGS, "-Wno-unused-parameter", "-shared", "-DUSE_ROCM", "-D__HIP_PLATFORM_AMD__=1",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f"-I{INCLUDE}",
            f"-I{sysconfig.get_paths()['include']}", f"-isystem{root / 'include'}",
            f"-isystem{root / 'include/torch/csrc/api/include'}", f"-isystem{_rocm() / 'include'}",
            str(CSRC / "gdnr_host.cpp"), "-o", str(out), f"-L{root / 'lib'}", "-ltorch_python", "-ltorch_cpu", "-lc10",
            "-lc10_hip"]


def build(verbose: bool = False) -> Path:
    BUILD_DIR.mkdir(exist_ok=True)
    inc = [f"-I{INCLUDE}", f"-I{CSRC}"]
    kern_objs, jobs = [], []
    for src in KERNEL_SOURCES:
        for i, act in enumerate(ACTS):
            obj = BUILD_DIR / f"{src}_{act}.o"
            kern_objs.append(obj)
            jobs.append([HIPCC, *DEVICE_FLAGS, *SOURCE_FLAGS.get(src, []), *inc, f"-DGDNR_ACT={i}", "-c",
                         str(CSRC / f"{src}.hip"), "-o", str(obj)])
    for src in SINGLE_SOURCES:
        obj = BUILD_DIR / f"{src}.o"
        kern_objs.append(obj)
        jobs.append([HIPCC, *DEVICE_FLAGS, *inc, "-c", str(CSRC / f"{src}.hip"), "-o", str(obj)])
    abi_obj = BUILD_DIR / "gdnr_abi.o"
    jobs.append(["g++", *HOST_FLAGS, *inc, "-c", str(CSRC / "gdnr_abi.cpp"), "-o", str(abi_obj)])
    host_tmp = HOST_MODULE.with_name(HOST_MODULE.name + ".tmp")
    with ThreadPoolExecutor(max_workers=len(jobs) + 1) as pool:
        # the library needs neither torch nor the module: a host without torch's
        # or Python's headers still gets it
        try:
            host_module = pool.submit(_run, _host_module_job(host_tmp), verbose)
        except ImportError:
            host_module = None
            print(f"torch is not importable: {HOST_MODULE.name} is not built", file=sys.stderr)
        for future in [pool.submit(_run, cmd, verbose) for cmd in jobs]:
            future.result()
    tmp = LIBRARY.with_name(LIBRARY.name + ".tmp")
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, kern_objs), str(abi_obj), "-o", str(tmp)],
         verbose)
    tmp.replace(LIBRARY)
    if host_module:
        host_module.result()
        host_tmp.replace(HOST_MODULE)
    return LIBRARY


def device_assembly(act: str = "bf16", src: str = "gdnr_step", out: Path | None = None,
                    verbose: bool = False) -> Path:
    """Write the gfx950 assembly of one source file's kernels for one
    activation dtype (inspection of waits, VGPR counts, instruction mix)."""
    out = out or BUILD_DIR / f"{src}_{act}.s"
    BUILD_DIR.mkdir(exist_ok=True)
    _run([HIPCC, *DEVICE_FLAGS, *SOURCE_FLAGS.get(src, []), f"-I{INCLUDE}", f"-I{CSRC}",
          f"-DGDNR_ACT={ACTS.index(act)}", "--cuda-device-only", "-S", str(CSRC / f"{src}.hip"), "-o", str(out)], verbose)
    return out


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
