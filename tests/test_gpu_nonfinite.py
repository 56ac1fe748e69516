"""Fields that overflow: infinities and NaN spread through the several-level sweep as through single
steps, walls and other solid voxels included (their value is 0 times what surrounds them)."""
import numpy as np
import pytest

import oracle
from parallelfdtd_amd import native as N
from parallelfdtd_amd import rooms
from parallelfdtd_amd.solver import Solver

pytestmark = pytest.mark.gpu

RAW = {N.F32: np.float32, N.F64: np.float64, N.F16: np.float16, N.BF16: np.uint16}
STEPS = 60


def walled(dims, n_boxes=4, seed=1300):
    """A room cut by thick walls whose rows are solid over whole tiles, along y and along z, with the
    source beside them."""
    X, Y, Z = dims
    sc = rooms.scene_random_small(seed, dims=dims, n_mat=4, n_boxes=n_boxes, n_src=2, n_rec=24, n_steps=STEPS)
    sc.labels[1:Z - 1, Y // 3:Y // 3 + min(30, Y // 4), X // 20:X - 8] = 2
    sc.labels[Z // 2:Z // 2 + max(3, Z // 8), 3:Y - 6, X // 8:X - X // 9] = 3
    sc.src_xyz[0] = [X // 2, Y // 3 - 2, Z // 2 - 2]
    sc.src_xyz[1] = [X // 3, Y // 3 + 3, Z // 3]  # inside the wall
    rng = np.random.default_rng(seed)
    near = np.repeat(sc.src_xyz, 12, axis=0)
    sc.rec_xyz = np.clip(near + rng.integers(-18, 19, near.shape), 1, np.array(dims) - 2).astype(np.int32)
    return sc


def f32(sig):
    return np.where(np.isfinite(sig), np.clip(sig, -3e38, 3e38), sig).astype(np.float32)


def run(sc, prec, levels, scale, signals, centred=False, zchunk=0, poll=100):
    with Solver() as s:
        if centred:
            s.set_update_type(N.SRL)
        s.set_time_levels(levels, zchunk)
        s.load_scene(sc)
        s.set_sources(sc.src_xyz, np.ones(len(sc.src_xyz), np.int32), signal_f64=signals.astype(np.float64),
                      signal_f32=f32(signals))
        s.set_poll_interval(poll)
        s.prepare_fields(prec, scale)
        s.run(STEPS, prec)
        return (s.responses(), *s.fields_raw(RAW[prec]))


def overflowing(prec, how):
    """(signals, storage scale): sums that pass the largest value, or an infinite or NaN sample."""
    sig = np.zeros((2, STEPS))
    if how == "sum":
        sig[0, :15] = {N.F64: 1e308, N.F16: 1.9}.get(prec, 3e38)
        return sig, 16 if prec == N.F16 else 0
    sig[:, :15] = 1.0
    sig[0 if how == "inf" else 1, 6] = {"inf": np.inf, "nan in the wall": np.nan}[how]
    return sig, 4 if prec in (N.F16, N.BF16) else 0


def values(a):
    return (a.astype(np.uint32) << 16).view(np.float32) if a.dtype == np.uint16 else a  # BF16 fields


def checked(out):
    """Bad values in some of the voxels and responses, the same ones on both sides."""
    assert 0 < (~np.isfinite(values(out[1][1]))).mean() < 1 and not np.isfinite(out[1][0]).all()
    for a, b in zip(*out):
        assert np.array_equal(values(a), values(b), equal_nan=True)


# rooms of the small tile, and of the large one (four fields above 256 MB)
SIZES = {"small": {p: (200, 100, 50) for p in RAW},
         "large": {N.F32: (400, 230, 200), N.F64: (300, 200, 150), N.F16: (540, 300, 220), N.BF16: (540, 300, 220)}}


@pytest.mark.parametrize("how", ["sum", "inf", "nan in the wall"])
@pytest.mark.parametrize("tile", list(SIZES))
@pytest.mark.parametrize("prec", list(RAW))
def test_overflow_as_with_single_steps(gpu, prec, tile, how):
    dims = SIZES[tile][prec]
    es = {N.F32: 4, N.F64: 8}.get(prec, 2)
    assert (4 * es * np.prod(dims) > 256 << 20) == (tile == "large")
    sc = walled(dims)
    sig, scale = overflowing(prec, how)
    out = [run(sc, prec, levels, scale, sig) for levels in (0, 1)]
    checked(out)


@pytest.mark.parametrize("zchunk,poll", [(3, 100), (0, 7)])
@pytest.mark.parametrize("prec", list(RAW))
def test_overflow_in_short_chunks_and_bundles(gpu, prec, zchunk, poll):
    sc = walled((260, 90, 40))
    sig, scale = overflowing(prec, "sum")
    out = [run(sc, prec, levels, scale, sig, zchunk=zchunk, poll=poll) for levels in (0, 1)]
    checked(out)


@pytest.mark.parametrize("tile", list(SIZES))
@pytest.mark.parametrize("prec", list(RAW))
def test_overflow_with_centred_boundaries(gpu, prec, tile):
    sc = walled(SIZES[tile][prec], n_boxes=0)
    sig, scale = overflowing(prec, "sum")
    out = [run(sc, prec, levels, scale, sig, centred=True) for levels in (0, 1)]
    checked(out)


@pytest.mark.parametrize("how", ["sum", "nan in the wall"])
@pytest.mark.parametrize("dims", [(200, 100, 50), (540, 300, 220)])
def test_overflow_of_the_difference_form(gpu, dims, how):
    """The oracle's difference form."""
    sc = walled(dims)
    sig, scale = overflowing(N.F16, how)
    pos, mat, _ = oracle.classify(sc.labels)
    ref = oracle.run(pos, mat, sc.material_table(), sc.src_xyz, np.ones(2, np.int32), sig.astype(np.float32),
                     sc.rec_xyz, STEPS, storage=oracle.STORE_F16_DIFF, scale_exp=scale, want_fields=True, threads=8)
    with Solver() as s:
        s.load_scene(sc)
        s.set_sources(sc.src_xyz, np.ones(2, np.int32), signal_f64=sig, signal_f32=f32(sig))
        s.prepare_fields(N.F16_DIFF, scale)
        s.run(STEPS, N.F16_DIFF)
        got = (s.responses(np.float32), *(f.astype(np.float32) for f in s.fields_raw(np.float16)))
    checked((got, ref))
