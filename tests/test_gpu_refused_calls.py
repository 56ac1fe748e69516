"""A refused call leaves the fields of a batch, their arrangement and the responses as they were: the
steps after it go on as if it had not been made."""
import numpy as np
import pytest

from parallelfdtd_amd import native as N
from parallelfdtd_amd import rooms
from parallelfdtd_amd.solver import Solver

pytestmark = pytest.mark.gpu

STEPS, B = 14, 4
REFUSED = {
    "prepare: FP32 takes no scale": lambda s: s.prepare_fields(N.F32, 3),
    "prepare: scale out of range": lambda s: s.prepare_fields(N.F16, 99),
    "prepare: unknown precision": lambda s: s.prepare_fields(77, 0),
    "run: unknown precision": lambda s: s.run(STEPS, 77),
    "begin: unknown precision": lambda s: s.begin_steps(STEPS, 77),
    "run: the difference form takes no batch": lambda s: s.run(STEPS, N.F16_DIFF),
}


def solver(prec, layout, seed=1100):
    sc = rooms.scene_random_small(seed, dims=(70, 44, 17), n_mat=3, n_boxes=3, n_src=B, n_rec=2 * B,
                                  n_steps=STEPS)
    s = Solver()
    s.load_scene(sc)
    s.set_batch_layout(layout)
    s.set_batch(B)
    s.set_source_slots(np.arange(B))
    s.set_receiver_slots(np.arange(2 * B) % B)
    if prec != N.F32:
        s.prepare_fields(prec, 9)
    return s


def outputs(s, prec):
    return (s.responses(), *s.fields_raw(np.float32 if prec == N.F32 else np.float16))


@pytest.mark.parametrize("what", list(REFUSED))
@pytest.mark.parametrize("prec", [N.F32, N.F16])
@pytest.mark.parametrize("layout", [N.BATCH_INTERLEAVED, N.BATCH_GROUPED])
def test_steps_go_on_after_a_refused_call(gpu, layout, prec, what):
    out = []
    for refuse in (False, True):
        with solver(prec, layout) as s:
            s.begin_steps(STEPS, prec)
            for k in range(STEPS):
                if refuse and k == 6:
                    with pytest.raises(N.PfdtdError):
                        REFUSED[what](s)
                s.step(k)
            out.append(outputs(s, prec))
    assert np.abs(out[0][0]).max() > 0
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("what", list(REFUSED))
@pytest.mark.parametrize("prec", [N.F32, N.F16])
def test_fields_of_a_run_after_a_refused_call(gpu, prec, what):
    """The default layout after a run, whose fields are held slot by slot."""
    with solver(prec, N.BATCH_INTERLEAVED) as s:
        s.run(STEPS, prec)
        before = outputs(s, prec)
        with pytest.raises(N.PfdtdError):
            REFUSED[what](s)
        after = outputs(s, prec)
        s.run(STEPS, prec)
        again = outputs(s, prec)
    assert np.abs(before[1]).max() > 0
    for a, b, c in zip(before, after, again):
        assert np.array_equal(a, b) and np.array_equal(a, c)
