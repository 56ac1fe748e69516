"""The several-level sweep keeps its rows in registers: the code objects of the built library say how much
memory a lane of each kernel takes besides (a loop left rolled up, or an array indexed at run time, moves
the queue there and slows the kernel to a third)."""
import re
import subprocess
from pathlib import Path

import pytest

from parallelfdtd_amd import native

LLVM = Path("/opt/rocm/llvm/bin")


def kernels(tmp_path):
    """{kernel name: (private bytes per lane, spilled vector registers)} of the library."""
    fat = tmp_path / "fat"
    subprocess.run([LLVM / "llvm-objcopy", f"--dump-section=.hip_fatbin={fat}", native.LIB_PATH, tmp_path / "lib"],
                   check=True)
    out = {}
    # a bundle per source, one after another
    data = fat.read_bytes()
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    starts = [m.start() for m in re.finditer(magic, data)]
    for i, (a, b) in enumerate(zip(starts, starts[1:] + [len(data)])):
        part, obj = tmp_path / f"bundle{i}", tmp_path / f"code{i}"
        part.write_bytes(data[a:b])
        subprocess.run([LLVM / "clang-offload-bundler", "--type=o", "--unbundle", f"--input={part}", f"--output={obj}",
                        "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True)
        notes = subprocess.run([LLVM / "llvm-readelf", "--notes", obj], check=True, capture_output=True,
                               text=True).stdout
        for entry in notes.split("- .agpr_count")[1:]:
            f = {k: v for k, v in re.findall(r"^\s+\.(name|private_segment_fixed_size|vgpr_spill_count):\s+(\S+)", entry,
                                             re.M)}
            out[re.findall(r"^    \.name:\s+(\S+)", entry, re.M)[-1]] = (int(f["private_segment_fixed_size"]),
                                                                       int(f["vgpr_spill_count"]))
    return out


def test_sweep_rows_stay_in_registers(tmp_path):
    if not (LLVM / "clang-offload-bundler").exists():
        pytest.skip("no ROCm tools")
    sweeps = {k: v for k, v in kernels(tmp_path).items() if "srl_sweep" in k}
    assert len(sweeps) >= 35, sorted(sweeps)
    worst = {k: v for k, v in sweeps.items() if v[0] > 64 or v[1] > 8}
    assert not worst, worst
