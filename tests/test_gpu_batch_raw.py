"""Reading the fields of a batch between its run and the steps that continue it changes nothing."""
import numpy as np
import pytest

from parallelfdtd_amd import native as N
from parallelfdtd_amd import rooms
from parallelfdtd_amd.solver import Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,dims", [(2, (57, 33, 12)), (8, (40, 60, 9))])
@pytest.mark.parametrize("prec,raw", [(N.F32, np.float32), (N.F16, np.float16)])
def test_steps_after_reading_the_fields_of_a_run(gpu, prec, raw, B, dims):
    sc = rooms.scene_random_small(1200, dims=dims, n_mat=3, n_boxes=2, n_src=B, n_rec=2 * B, n_steps=20)
    out = []
    for read in (False, True):
        with Solver() as s:
            s.load_scene(sc)
            s.set_batch(B)
            s.set_source_slots(np.arange(B))
            s.set_receiver_slots(np.arange(2 * B) % B)
            s.prepare_fields(prec, 9 if prec == N.F16 else 0)
            s.run(20, prec)
            if read:
                first, again = s.fields_raw(raw), s.fields_raw(raw)
                assert np.abs(first[0]).max() > 0
                assert all(np.array_equal(a, b) for a, b in zip(first, again))
            s.steps(3, 11)
            out.append((s.responses(), *s.fields_raw(raw)))
    assert np.abs(out[0][0]).max() > 0
    for a, b in zip(*out):
        assert np.array_equal(a, b)
