"""The serving pool's host code on the stand-in HIP runtime: the launch tables it builds."""
import numpy as np
import pytest

import hostrt
from parallelfdtd_amd import native as N
from parallelfdtd_amd import rooms
from parallelfdtd_amd import serve as S


@pytest.fixture(scope="module")
def rt(tmp_path_factory):
    r = hostrt.Runtime(hostrt.build(tmp_path_factory.mktemp("hostrt")))
    kept, N._lib = N._lib, r.lib
    yield r
    N._lib = kept


def job(dims, n_steps, boundary_source=False, precision=N.F32):
    sc = rooms.scene_random_small(7, dims=dims, n_mat=2, n_boxes=0, n_src=2, n_rec=2, n_steps=n_steps)
    src = sc.src_xyz.copy()
    if boundary_source:
        src[0, 2] = 0
    return S.JobSpec(sc.labels, np.array([0.1, 0.2], np.float32), src, np.ones(2, np.int32),
                     sc.signals.astype(np.float32), sc.rec_xyz, n_steps, precision)


@pytest.mark.parametrize("precision", [N.F32, N.F16, N.BF16])
@pytest.mark.parametrize("large_first", [True, False])
def test_sweep_blocks_of_rooms_beside_single_step_jobs(rt, precision, large_first):
    """A job of single steps (a source on slice 0) beside jobs of the sweep of another size: every job
    of the sweep is launched with the blocks of its own room."""
    big, small = (150, 100, 90), (20, 16, 12)
    a, b = (big, small) if large_first else (small, big)
    with S.Pool(0, arena_bytes=1 << 28, bundle=5) as pool:
        for spec in (job(a, 50, precision=precision), job(b, 40, True, precision), job(b, 45, precision=precision),
                     job(a, 35, True, precision)):
            assert pool.submit(spec) is not None
            rt.log()
            pool.advance()
            sweeps = [l for l in rt.log() if l.startswith("pool_sweep")]
            assert sweeps and all(l.endswith("bad=none") for l in sweeps), sweeps
