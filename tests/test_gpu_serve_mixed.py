"""Jobs of single steps (a source on the never-updated first z slice) beside jobs of the several-level
sweep, rooms of different sizes in either order of submission: each equals the job alone."""
import numpy as np
import pytest

from parallelfdtd_amd import native as N
from parallelfdtd_amd import rooms
from parallelfdtd_amd import serve as S
from test_gpu_serve import drive

pytestmark = pytest.mark.gpu


def job(seed, dims, n_steps, precision, boundary_source):
    sc = rooms.scene_random_small(seed, dims=dims, n_mat=3, n_boxes=3, n_src=2, n_rec=4, n_steps=n_steps)
    src, rec = sc.src_xyz.copy(), sc.rec_xyz.copy()
    if boundary_source:
        src[0, 2] = 0
    for k in range(len(rec) - 1):  # near the sources, so that they hear them in time
        rec[k] = np.minimum(src[k % 2] + [1 + k, 1, 1], np.array(dims) - 2)
    return S.JobSpec(sc.labels, np.array([0.1, 0.3, 0.5], np.float32), src, np.ones(2, np.int32),
                     sc.signals.astype(np.float32), rec, n_steps, precision,
                     9 if precision != N.F32 else 0)


@pytest.mark.parametrize("precision", [N.F32, N.F16, N.BF16])
@pytest.mark.parametrize("large_first", [True, False])
def test_rooms_of_two_sizes_beside_single_step_jobs(gpu, precision, large_first):
    big, small = (150, 100, 90), (34, 30, 22)
    a, b = (big, small) if large_first else (small, big)
    specs = [job(31, a, 123, precision, False), job(32, b, 60, precision, True),
             job(33, b, 77, precision, False), job(34, a, 40, precision, True)]
    alone = [S.run_alone(j) for j in specs]
    with S.Pool(0, arena_bytes=1 << 30, bundle=10) as pool:
        got = drive(pool, specs, schedule=[0, 1, 2, 3])
    for k, j in enumerate(specs):
        assert np.abs(alone[k]).max() > 0
        assert np.array_equal(got[k], alone[k]), f"job {k} ({j.labels.shape}, {j.n_steps} steps)"
