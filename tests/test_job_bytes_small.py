"""The size query of a serving job answers for rooms the pool would refuse too (fewer than three
slices), and grows with the room. In a process of its own: a crash would end it."""
import subprocess
import sys

import pytest

SCRIPT = """
import ctypes, sys
from parallelfdtd_amd import native as N
sizes = []
for Z in (1, 2, 3, 4):
    j = N.PfdtdJob(X=int(sys.argv[1]), Y=int(sys.argv[2]), Z=Z, n_src=0, n_samples=0, n_rec=1, n_steps=4,
                   precision=int(sys.argv[3]))
    b = ctypes.c_int64(-1)
    assert N.lib().pfdtd_pool_job_bytes(ctypes.byref(j), ctypes.byref(b)) == N.OK
    sizes.append(b.value)
print(*sizes)
"""


@pytest.mark.parametrize("precision", [0, 2, 3])
@pytest.mark.parametrize("X,Y", [(1, 1), (3, 2), (40, 30), (2147483647, 1)])
def test_job_bytes_of_thin_rooms(X, Y, precision):
    out = subprocess.run([sys.executable, "-c", SCRIPT, str(X), str(Y), str(precision)],
                         capture_output=True, text=True)
    assert out.returncode == 0, (out.returncode, out.stderr)
    sizes = [int(v) for v in out.stdout.split()]
    es = 4 if precision == 0 else 2
    for z, b in zip((1, 2, 3, 4), sizes):
        # two fields and three byte planes, for the sweep two more fields and the entry plane
        swept = X * Y * es < 2 ** 31
        assert (4 * es + 5 if swept else 2 * es + 3) * X * Y * z <= b < 2 ** 50
    assert sizes == sorted(sizes)
