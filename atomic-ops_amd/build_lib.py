"""Build ``libgdn2_hip.so`` in-tree with hipcc for gfx950, and the native call path ``_bind.so``
(host C++ against this torch) with g++.

Usage: ``python atomic-ops_amd/build_lib.py`` (also called by ``__graft_entry__.build()``).
Each ``csrc/*.hip`` translation unit is compiled to an object in ``_build/`` in parallel,
then linked into ``atomic_gdn2/_lib/libgdn2_hip.so`` next to the Python package.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
from pathlib import Path

HERE = Path(__file__).resolve().parent
CSRC = HERE / "csrc"
BUILD = HERE / "_build"
OUT = HERE / "atomic_gdn2" / "_lib" / "libgdn2_hip.so"
ARCH = os.environ.get("GDN2_OFFLOAD_ARCH", "gfx950")

# -packed-fp32-ops: keep the compiler from emitting packed fp32 VALU ops.
# -amdgpu-mfma-vgpr-form: keep MFMA accumulators in VGPRs.  With accumulators in AGPRs the
#   compiler placed ~8 wait states between the last v_mfma_f32_16x16x4_f32 of a chain and the
#   v_accvgpr_read of its 4th result register, and that register came back stale on gfx950
#   (only accumulator element 3 wrong, only where the last k-step contributes).
HIPFLAGS = [
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-mllvm", "-amdgpu-mfma-vgpr-form=1",
    "-Wall", "-Wno-unused-function", "-Wno-unused-variable",
    f"-I{HERE.parent / 'include'}",
]


def _hipcc() -> str:
    p = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(p).exists():
        raise RuntimeError("hipcc not found; the HIP library cannot be built")
    return p


def _compile(src: Path, verbose: bool) -> Path:
    obj = BUILD / (src.stem + ".o")
    cmd = [_hipcc(), *HIPFLAGS, "-c", str(src), "-o", str(obj)]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    msgs = "\n".join(l for l in (r.stdout + r.stderr).splitlines()
                     if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src.name}:\n{msgs}")
    if verbose and msgs.strip():
        print(msgs, flush=True)
    return obj


def _build_bind(verbose: bool) -> Path:
    import sysconfig

    import torch
    from torch.utils import cpp_extension
    out = HERE / "atomic_gdn2" / "_bind.so"
    tmp = BUILD / "_bind.so.tmp"
    lib = Path(torch.__file__).resolve().parent / "lib"
    rocm = Path(os.environ.get("ROCM_PATH", "/opt/rocm"))
    incs = [*cpp_extension.include_paths(), sysconfig.get_paths()["include"], str(rocm / "include")]
    cmd = [shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-w",
           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *(f"-I{i}" for i in incs), str(CSRC / "bind.cpp"), "-o", str(tmp), f"-L{lib}", f"-Wl,-rpath,{lib}",
           "-Wl,--no-as-needed", "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-ltorch", "-ltorch_python"]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed on bind.cpp:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, out)
    return out


def build(verbose: bool = False) -> Path:
    BUILD.mkdir(exist_ok=True)
    OUT.parent.mkdir(parents=True, exist_ok=True)
    srcs = sorted(CSRC.glob("*.hip"))
    with cf.ThreadPoolExecutor(max_workers=8) as ex:
        bind = ex.submit(_build_bind, verbose)
        objs = list(ex.map(lambda s: _compile(s, verbose), srcs))
        bind.result()
    tmp = OUT.with_suffix(".so.tmp")
    cmd = [_hipcc(), "-shared", "-fPIC", f"--offload-arch={ARCH}", *map(str, objs), "-o", str(tmp)]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, OUT)
    return OUT


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
