"""Builds a kernel source for the host (tests/native/host_hip), where it runs
with its waves and lanes in a chosen order."""
import ctypes
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
CSRC = ROOT / "glm-5.3-kernels_amd" / "csrc"


def build(source: str, folder: Path) -> ctypes.CDLL:
    """csrc/<source> as a host library, built in `folder`."""
    clang = shutil.which("clang++", path="/opt/rocm/llvm/bin") or shutil.which("clang++")
    if clang is None:
        pytest.skip("clang++ not available")
    lds_barrier = 'asm volatile("s_waitcnt lgkmcnt(0)\\n\\ts_barrier" ::: "memory")'
    for name, to in ((source, "kernel.cpp"), ("glm53_common.h", "glm53_common.h")):
        text = (CSRC / name).read_text().replace(lds_barrier, "host_hip::barrier(0)")
        (folder / to).write_text(text.replace("__builtin_amdgcn_", "host_amdgcn_"))
    lib = folder / "libhost.so"
    subprocess.run([clang, "-O1", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-w", f"-I{folder}",
                    f"-I{ROOT / 'tests' / 'native' / 'host_hip'}", f"-I{ROOT / 'include'}",
                    str(folder / "kernel.cpp"), "-o", str(lib)], check=True)
    return ctypes.CDLL(str(lib))
