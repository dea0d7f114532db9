"""The operators' .hip sources compiled for the CPU (tests/cpp/lockstep): their C ABI over host memory, with
the kernels run one workgroup after another and the waves of each as unevenly as its barriers allow."""
from __future__ import annotations

import concurrent.futures as cf
import ctypes
import os
import subprocess
from pathlib import Path
from typing import NamedTuple

import numpy as np

from ahead_amd import an, capi

ROOT = Path(__file__).resolve().parents[1]
HERE = ROOT / "tests" / "cpp" / "lockstep"
OUT = ROOT / "tests" / "cpp" / "_build" / "lockstep"
CXX = Path("/opt/rocm/llvm/bin/clang++")
UNITS = ["runtime", "decode_an", "ops_an", "ops2_an", "merge_an", "groupby_an", "hashjoin_an"]

_lib = None


def available() -> bool:
    return CXX.exists()


def _sources():
    csrc = ROOT / "ahead_amd" / "csrc"
    return [csrc / f"{u}.hip" for u in UNITS] + [HERE / "lockstep.cpp"]


def build() -> Path:
    OUT.mkdir(parents=True, exist_ok=True)
    so = OUT / "liblockstep.so"
    deps = _sources() + sorted((ROOT / "ahead_amd" / "csrc").glob("*.hpp")) + [HERE / "hip" / "hip_runtime.h",
                                                                              ROOT / "include" / "ahead_hip.h"]
    if so.exists() and all(d.stat().st_mtime < so.stat().st_mtime for d in deps):
        return so

    def compile_(src: Path) -> str:
        obj = OUT / f"{src.stem}.{os.getpid()}.o"
        subprocess.run([str(CXX), "-x", "c++", "-std=c++17", "-O1", "-fPIC", "-Wno-unknown-attributes", f"-I{HERE}",
                        f"-I{ROOT / 'include'}", "-c", str(src), "-o", str(obj)], check=True)
        return str(obj)
    with cf.ThreadPoolExecutor(max_workers=4) as ex:
        objs = list(ex.map(compile_, _sources()))
    tmp = OUT / f"liblockstep.{os.getpid()}.tmp"
    subprocess.run([str(CXX), "-shared", "-o", str(tmp), *objs], check=True)
    for o in objs:
        os.unlink(o)
    os.replace(tmp, so)
    return so


def lib() -> ctypes.CDLL:
    global _lib
    if _lib is None:
        L = ctypes.CDLL(str(build()))
        for name, (args, res) in capi._SIGS.items():
            if hasattr(L, name):
                fn = getattr(L, name)
                fn.argtypes, fn.restype = args, res
        L.lockstep_set.argtypes = [ctypes.c_int] * 3
        L.lockstep_launches.restype = ctypes.c_char_p
        _lib = L
    return _lib


def check(st: int) -> None:
    if st:
        raise RuntimeError(f"status {st}: {lib().ahead_hip_last_error().decode()}")


class Workspace:
    def __init__(self, device: int = 0):
        self.h = ctypes.c_void_p()
        check(lib().ahead_hip_ws_create(device, ctypes.byref(self.h)))

    def bytes(self) -> int:
        return int(lib().ahead_hip_ws_bytes(self.h))

    def __del__(self):
        lib().ahead_hip_ws_destroy(self.h)


class Launch(NamedTuple):
    kernel: str
    grid: int
    block: int
    steps: int  # wave-wide operations and barriers its waves went through
    swaps: int  # compare-and-swaps its lanes made


def launches() -> list[Launch]:
    """Every launch since the last call; ("attribute", device, 0, 0, 0) for each hipFuncSetAttribute."""
    out = []
    for line in lib().lockstep_launches().decode().splitlines():
        if line.startswith("attribute"):
            out.append(Launch("attribute", int(line.split()[1]), 0, 0, 0))
        else:
            name, *v = line.rsplit(" ", 4)
            out.append(Launch(name.strip("()"), *map(int, v)))
    return out


def column(arr: np.ndarray | None, meta: an.ColMeta, n: int | None = None, seqbase: int = 0, data: int | None = None):
    """An ahead_col over a host array (None: void), or over `data` as it stands (a launch that is not run)."""
    t = meta.type
    c = capi.AheadCol()
    c.data = (arr.ctypes.data if arr is not None else None) if data is None else data
    c.n = len(arr) if n is None else n
    c.width, c.encoded, c.unenc_bits = t.width, int(t.encoded), t.unenc_bits
    c.a, c.a_inv, c.max_u, c.seqbase = meta.a, meta.a_inv, t.max_u, seqbase or meta.seqbase
    c._keep = arr
    return c


def buf(arr: np.ndarray) -> capi.Buf:
    return capi.Buf(arr.ctypes.data, len(arr))
