"""The library's host code on a stand-in HIP runtime (fake_hip.cpp): what it allocates, launches and
refuses, on the CPU. Kernels do not run, so fields and responses stay zero."""
from __future__ import annotations

import ctypes as C
import re
import subprocess
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

from parallelfdtd_amd import build as B
from parallelfdtd_amd import native as N

HERE = Path(__file__).resolve().parent
UNDEFINED_IMAGE = re.compile(r"\bU (__hip_fatbin\w*)")


def _objects(sources: list[Path], out: Path) -> list[str]:
    """The host half of HIP sources, compiled."""
    flags = [B.HIPCC, "--offload-arch=gfx950", "--cuda-host-only", "-O1", "-std=c++17", "-fPIC",
             "-I", str(B.ROOT / "include"), "-I", str(B.CSRC)]

    def one(src: Path) -> str:
        obj = out / (src.stem + ".o")
        subprocess.run([*flags, "-x", "hip", "-c", str(src), "-o", str(obj)], check=True)
        return str(obj)

    with ThreadPoolExecutor(8) as ex:
        return list(ex.map(one, sources))


def _no_images(objs: list[str]) -> list[str]:
    """No device images: the symbols that would name them are absolute zeros."""
    names = subprocess.run(["nm", "-u", *objs], check=True, capture_output=True, text=True).stdout
    return [f"-Wl,--defsym={s}=0" for s in sorted(set(UNDEFINED_IMAGE.findall(names)))]


def build(out: Path) -> Path:
    """libpfdtd with the host half of every source only, linked to the stand-in runtime."""
    objs = _objects([*(B.CSRC / s for s in B.LIB_SOURCES), HERE / "fake_hip.cpp"], out)
    lib = out / "libpfdtd_host.so"
    subprocess.run(["g++", "-shared", "-fPIC", "-Wl,-Bsymbolic", "-o", str(lib), *objs, *_no_images(objs)],
                   check=True)
    return lib


def run_program(source: str, uses: list[str], out: Path) -> subprocess.CompletedProcess:
    """A program over the library's host functions, with the named sources of it, run to its end."""
    main = out / "program.hip"
    main.write_text(source)
    objs = _objects([main, HERE / "fake_hip.cpp", *(B.CSRC / u for u in uses)], out)
    exe = out / "program"
    # launchers of other sources are not called: their symbols may stay unresolved
    subprocess.run(["g++", "-no-pie", *objs, *_no_images(objs), "-Wl,--unresolved-symbols=ignore-all",
                    "-o", str(exe)], check=True)
    return subprocess.run([str(exe)], capture_output=True, text=True)


class Runtime:
    """The loaded library and the stand-in runtime's controls."""

    def __init__(self, path: Path):
        self.lib = C.CDLL(str(path))
        for name, args in N.SIGNATURES.items():
            fn = getattr(self.lib, name)
            fn.argtypes = args
            fn.restype = N._RESTYPE.get(name, C.c_int)
        self.lib.fake_budget.argtypes = [C.c_size_t]
        self.lib.fake_used.restype = C.c_size_t
        self.lib.fake_log_line.restype = C.c_char_p

    def fail_malloc(self, n: int) -> None:
        self.lib.fake_fail_malloc(n)

    def budget(self, n: int) -> None:
        self.lib.fake_budget(n)

    def used(self) -> int:
        return self.lib.fake_used()

    def log(self) -> list[str]:
        """The launches since the last call."""
        lines = [self.lib.fake_log_line(i).decode() for i in range(self.lib.fake_log_lines())]
        self.lib.fake_clear_log()
        return lines
