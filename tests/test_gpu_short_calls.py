"""Calls of one, two and a few steps, whichever kernels they take, continue each other: responses and
fields are those of single steps. Rooms of the large tile, at sizes on both sides of the lines."""
import numpy as np
import pytest

from parallelfdtd_amd import native as N
from parallelfdtd_amd import rooms
from parallelfdtd_amd.solver import Solver

pytestmark = pytest.mark.gpu

RAW = {N.F32: np.float32, N.F64: np.float64, N.F16: np.float16, N.BF16: np.uint16}
STEPS = 31


@pytest.mark.parametrize("dims,prec,centred", [
    ((256, 256, 256), N.F32, False), ((384, 320, 200), N.F32, False), ((448, 264, 135), N.F32, True),
    ((384, 320, 200), N.F64, False), ((640, 480, 240), N.F64, False), ((256, 256, 256), N.F16, False),
    ((640, 480, 260), N.F16, False), ((255, 256, 256), N.BF16, False), ((1024, 768, 352), N.F16, False)])
def test_short_calls_continue_each_other(gpu, dims, prec, centred):
    X, Y, Z = dims
    lab = rooms.box_room(X, Y, Z, floor=0, ceiling=1, walls=2)
    if not centred:
        rooms.add_boxes(lab, rooms.SplitMix64(3), 6, 2, 20, [0, 1, 2])
    src = np.array([[X // 2, Y // 2, Z // 2], [X // 2 + 3, Y // 2, Z // 2]], np.int32)
    rec = np.array([[X // 2 + d, Y // 2 + 1, Z // 2 - 1] for d in range(-6, 7)], np.int32)
    sig = np.random.default_rng(1).uniform(-1, 1, (2, STEPS))
    out = []
    for levels in (1, 0):
        with Solver() as s:
            if centred:
                s.set_update_type(N.SRL)
            s.set_time_levels(levels)
            s.set_domain_labels(lab)
            s.set_materials(np.repeat(np.array([0.1, 0.3, 0.5], np.float32)[:, None], 20, axis=1))
            s.set_sources(src, np.ones(2, np.int32), signal_f64=sig, signal_f32=sig.astype(np.float32))
            s.set_receivers(rec)
            s.prepare_fields(prec, 9 if prec in (N.F16, N.BF16) else 0)
            got = []
            for poll in (100, 1, 2) if levels == 0 else (100,):
                s.set_poll_interval(poll)
                s.run(STEPS, prec)
                got.append((s.responses(), *s.fields_raw(RAW[prec])))
            s.begin_steps(STEPS, prec)
            k = 0
            for n in (1, 2, 1, 1, 2, 2, 6, 4, 1, 7, 3, 1):
                s.steps(k, n)
                k += n
            assert k == STEPS
            got.append((s.responses(), *s.fields_raw(RAW[prec])))
            out.append(got)
    ref = out[0][0]
    assert np.abs(ref[0]).max() > 0
    for got in out[0][1:] + out[1]:
        for a, b in zip(ref, got):
            assert np.array_equal(a, b)
