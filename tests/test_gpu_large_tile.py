"""The large tile of the several-level sweep in every mode: rooms one column or row either side of its
borders, events on the columns and rows that tiles share, chunks of few slices, remainders of the levels.
(That these rooms take the large tile is tested on the CPU.)"""
import numpy as np
import pytest

import oracle
from large_tile import BORDERS, scene
from parallelfdtd_amd import native as N
from parallelfdtd_amd.solver import Solver

pytestmark = pytest.mark.gpu

RAW = {N.F32: np.float32, N.F64: np.float64, N.F16: np.float16, N.BF16: np.uint16}


@pytest.mark.parametrize("dx,dy,zchunk,n_steps", BORDERS)
@pytest.mark.parametrize("centred", [False, True])
@pytest.mark.parametrize("prec", list(RAW))
def test_borders_agree_with_single_steps(gpu, prec, centred, dx, dy, zchunk, n_steps):
    sc = scene(prec, dx, dy, n_steps, centred)
    out = []
    for levels in (0, 1):
        with Solver() as s:
            if centred:
                s.set_update_type(N.SRL)
            s.set_time_levels(levels, zchunk)
            s.load_scene(sc)
            s.prepare_fields(prec, 9 if prec in (N.F16, N.BF16) else 0)
            s.run(n_steps, prec)
            out.append((s.responses(), *s.fields_raw(RAW[prec])))
    assert (np.abs(out[1][0]).max(axis=1) > 0).mean() > 0.2
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("dx,dy,zchunk,n_steps", BORDERS)
def test_borders_of_the_difference_form_agree_with_the_oracle(gpu, dx, dy, zchunk, n_steps):
    sc = scene(N.F16_DIFF, dx, dy, n_steps)
    pos, mat, _ = oracle.classify(sc.labels)
    ref = oracle.run(pos, mat, sc.material_table(), sc.src_xyz, sc.src_kind, sc.signals.astype(np.float32),
                     sc.rec_xyz, n_steps, storage=oracle.STORE_F16_DIFF, scale_exp=9, want_fields=True, threads=8)
    with Solver() as s:
        s.set_time_levels(0, zchunk)
        s.load_scene(sc)
        s.prepare_fields(N.F16_DIFF, 9)
        s.run(n_steps, N.F16_DIFF)
        got = (s.responses(np.float32), *(f.astype(np.float32) for f in s.fields_raw(np.float16)))
    assert (np.abs(ref[0]).max(axis=1) > 0).mean() > 0.2
    for a, b in zip(got, ref):
        assert np.array_equal(a, b)
