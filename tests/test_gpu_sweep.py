"""GPU parity of the several-level sweep (the automatic path of FP32 and FP64 runs) against the
CPU oracle at the sizes where it can go wrong: rooms one column or row either side of its tile
borders, the smallest rooms, chunks of few slices, every remainder of the step count, events on
tile borders and many to a tile. Bar: bit-identical responses and final fields."""
import numpy as np
import pytest

from parallelfdtd_amd import native as N
from parallelfdtd_amd import rooms
from parallelfdtd_amd.solver import Solver
from test_gpu_fused import assert_same, run_both

pytestmark = pytest.mark.gpu

OWNED = {N.F32: (112, 38), N.F64: (56, 56), N.F16: (112, 38), N.BF16: (112, 38)}  # owned columns and rows of a block


def scene(seed, dims, n_steps, n_boxes=6, n_src=3, n_rec=8):
    return rooms.scene_random_small(seed, dims=dims, n_mat=4, n_boxes=n_boxes, n_src=n_src,
                                    n_rec=n_rec, n_steps=n_steps)


@pytest.mark.parametrize("prec", list(OWNED))
@pytest.mark.parametrize("dx,dy,z,zchunk", [(-1, 1, 9, 0), (0, 0, 12, 3), (1, -1, 21, 5),
                                            (8, 5, 8, 1), (9, 6, 30, 7)])
def test_tile_borders(gpu, prec, dx, dy, z, zchunk):
    ox, oy = OWNED[prec]
    sc = scene(900 + dx, (ox + dx, 2 * oy + dy, z), 23, n_boxes=12)
    # sources and receivers in the columns and rows two neighbouring tiles share
    sc.src_xyz[0] = [ox - 3 if dx < 1 else ox - 1, oy, z // 2]
    sc.rec_xyz[0] = [min(ox, ox + dx - 2), oy - 1, z // 2]
    sc.rec_xyz[1] = sc.src_xyz[0]
    assert_same(*run_both(sc, prec, levels=0, zchunk=zchunk))


@pytest.mark.parametrize("prec", list(OWNED))
@pytest.mark.parametrize("n_steps", [1, 2, 3, 4, 5, 6, 9])
def test_step_remainders(gpu, prec, n_steps):
    assert_same(*run_both(scene(910, (131, 50, 17), n_steps), prec, levels=0, zchunk=0))


@pytest.mark.parametrize("prec", list(OWNED))
@pytest.mark.parametrize("dims", [(3, 3, 3), (4, 3, 5), (5, 90, 3), (301, 4, 4), (7, 5, 140)])
def test_small_and_thin_rooms(gpu, prec, dims):
    sc = scene(920, dims, 14, n_boxes=0, n_src=1, n_rec=3)
    assert_same(*run_both(sc, prec, levels=0, zchunk=0))


@pytest.mark.parametrize("prec", list(OWNED))
def test_many_events_in_one_tile(gpu, prec):
    """A plane of receivers, several sources on one voxel, hard and soft, on shell voxels too;
    bundles of 7 steps (5 and 2 levels)."""
    sc = scene(930, (64, 40, 12), 21, n_src=1)
    g = np.array([[x, y, 5] for y in range(3, 37) for x in range(2, 62)], np.int32)
    sc.rec_xyz = g
    sc.src_xyz = np.concatenate([g[100:130], g[100:103], [[0, 9, 5], [63, 9, 6], [20, 0, 4]]])
    sc.src_xyz = sc.src_xyz.astype(np.int32)
    sc.src_kind = np.array([i % 2 for i in range(len(sc.src_xyz))], np.int32)
    sc.signals = np.random.default_rng(5).uniform(-1, 1, (len(sc.src_xyz), sc.n_steps))
    with_poll = run_both(sc, prec, levels=0, zchunk=0, poll=7)
    assert_same(*with_poll)


@pytest.mark.parametrize("prec", list(OWNED))
def test_other_lambda_and_solid_regions(gpu, prec):
    """A room half solid (rows with nothing to update), sources inside the solid."""
    sc = scene(940, (150, 60, 40), 33)
    sc.labels[:, 22:, 70:] = 2
    sc.src_xyz[0] = [100, 40, 20]
    assert_same(*run_both(sc, prec, levels=0, zchunk=0))


def test_steps_and_captures_agree_with_run(gpu):
    """Segments of every length through pfdtd_steps give the run's responses."""
    sc = scene(950, (120, 45, 20), 60)
    with Solver() as s:
        s.load_scene(sc)
        s.run(sc.n_steps, N.F32)
        ref = s.responses(np.float32)
        s.begin_steps(sc.n_steps, N.F32)
        k, n = 0, 1
        while k < sc.n_steps:
            m = min(n, sc.n_steps - k)
            s.steps(k, m)
            k, n = k + m, n + 1
        assert np.array_equal(s.responses(np.float32), ref)


def test_changed_domain_sources_and_precision(gpu):
    """One context, re-used: the sweep's planes and events follow each change."""
    a, b = scene(960, (90, 44, 16), 12), scene(961, (44, 90, 16), 12)
    with Solver() as s, Solver() as t:
        for sc, prec in ((a, N.F32), (b, N.F64), (a, N.F64), (b, N.F32)):
            for x in (s,):
                x.load_scene(sc)
                x.run(sc.n_steps, prec)
            t.set_time_levels(1)
            t.load_scene(sc)
            t.run(sc.n_steps, prec)
            assert np.array_equal(s.responses(), t.responses())
            s.set_receivers(sc.rec_xyz[::-1].copy())
            s.run(sc.n_steps, prec)
            assert np.array_equal(s.responses()[::-1], t.responses())


@pytest.mark.parametrize("prec", list(OWNED))
@pytest.mark.parametrize("B,dims", [(2, (121, 39, 11)), (16, (50, 44, 9))])
def test_interleaved_batch_agrees_with_grouped_and_steps(gpu, prec, B, dims):
    """The default (interleaved) layout, whose runs hold the slots one after another: responses,
    interleaved raw fields, and step calls before and after a run."""
    sc = scene(970, dims, 13, n_src=B, n_rec=2 * B)
    raw = {N.F32: np.float32, N.F64: np.float64, N.F16: np.float16, N.BF16: np.uint16}[prec]
    scale = 9 if prec in (N.F16, N.BF16) else 0
    out = []
    for layout in (N.BATCH_INTERLEAVED, N.BATCH_GROUPED):
        with Solver() as s:
            s.load_scene(sc)
            s.set_batch_layout(layout)
            s.set_batch(B)
            s.set_source_slots(np.arange(B))
            s.set_receiver_slots(np.arange(2 * B) % B)
            s.prepare_fields(prec, scale)
            for _ in range(2):
                s.run(sc.n_steps, prec)
                r, (P, Pp) = s.responses(), s.fields_raw(raw)
                s.begin_steps(sc.n_steps, prec)
                for k in range(sc.n_steps):
                    s.step(k)
                assert np.array_equal(s.responses(), r)
            if layout == N.BATCH_INTERLEAVED:
                P, Pp = np.moveaxis(P, -1, 0), np.moveaxis(Pp, -1, 0)
            out.append((r, P, Pp))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    assert all(f.any() for f in out[0][1])  # every slot holds its own source


@pytest.mark.parametrize("dx,dy,z,zchunk", [(-2, 1, 9, 0), (0, -1, 12, 3), (2, 0, 21, 5), (8, 5, 8, 1)])
@pytest.mark.parametrize("n_steps", [23, 4])
def test_difference_form_at_tile_borders(gpu, dx, dy, z, zchunk, n_steps):
    """P and D of the difference form either side of a tile border, every remainder of the levels,
    sources in solid voxels and on two tiles' shared columns."""
    from test_gpu_diff import run_diff
    ox, oy = OWNED[N.F16]
    sc = scene(980 + dx, (ox + dx, 2 * oy + dy, z), n_steps, n_boxes=12)
    sc.src_xyz[0] = [ox - 3, oy, z // 2]
    sc.labels[z // 2, oy + 3, 5:9] = 1
    sc.src_xyz[1] = [6, oy + 3, z // 2]
    sc.rec_xyz[0] = sc.src_xyz[0]
    run_diff(sc, 9, zchunk=zchunk, poll=7)


@pytest.mark.parametrize("prec", list(OWNED))
@pytest.mark.parametrize("dx,dy,z,zchunk,n_steps", [(-1, 1, 9, 0, 23), (0, 0, 12, 3, 9), (1, -1, 21, 5, 7),
                                                    (9, 6, 30, 7, 14)])
def test_centred_scheme_agrees_with_single_steps(gpu, prec, dx, dy, z, zchunk, n_steps):
    """The centred boundaries through the sweep and through single steps, whose parity with the oracle
    is tested elsewhere: responses and both fields bit for bit."""
    from test_gpu_centred import centred_room
    ox, oy = OWNED[prec]
    sc = centred_room(1010 + dx, (ox + dx, 2 * oy + dy, z), n_steps=n_steps)
    sc.src_xyz[0] = [ox // 2, oy, 1]
    sc.rec_xyz[0] = [ox // 2 + 1, oy, 1]
    raw = {N.F32: np.float32, N.F64: np.float64, N.F16: np.float16, N.BF16: np.uint16}[prec]
    out = []
    for levels in (0, 1):
        with Solver() as s:
            s.set_update_type(N.SRL)
            s.set_time_levels(levels, zchunk)
            s.load_scene(sc)
            s.prepare_fields(prec, 9 if prec in (N.F16, N.BF16) else 0)
            s.run(sc.n_steps, prec)
            out.append((s.responses(), *s.fields_raw(raw)))
    assert out[1][1].any()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


SMALL = {N.F32: (56, 18), N.F64: (56, 26), N.F16: (56, 18), N.BF16: (56, 18)}  # of the small tile


@pytest.mark.parametrize("prec", list(SMALL))
@pytest.mark.parametrize("dx,dy,z,zchunk", [(-1, 1, 9, 0), (0, 0, 12, 3), (1, -1, 21, 5), (8, 5, 8, 1)])
@pytest.mark.parametrize("n_steps", [23, 4])
def test_small_tile_borders(gpu, prec, dx, dy, z, zchunk, n_steps):
    """Rooms the small tile takes: two tiles and a little more or less along x and y."""
    ox, oy = SMALL[prec]
    sc = scene(990 + dx, (2 * ox + dx, 2 * oy + dy, z), n_steps, n_boxes=12)
    sc.src_xyz[0] = [ox - 3, oy, z // 2]
    sc.rec_xyz[0] = [ox, oy - 1, z // 2]
    sc.rec_xyz[1] = sc.src_xyz[0]
    assert_same(*run_both(sc, prec, levels=0, zchunk=zchunk))


@pytest.mark.parametrize("prec", list(OWNED))
@pytest.mark.parametrize("dims", [(331, 150, 60), (224, 113, 97)])
def test_large_tile_agrees_with_single_steps(gpu, prec, dims):
    """Enough sources at once for the large tile, several tiles along x and y, each slot its own
    source, against single steps of the same batch."""
    B = 8
    sc = scene(1000, dims, 19, n_boxes=20, n_src=B, n_rec=4 * B)
    out = []
    for levels in (0, 1):
        with Solver() as s:
            s.set_time_levels(levels, 0)
            s.load_scene(sc)
            s.set_batch_layout(N.BATCH_GROUPED)
            s.set_batch(B)
            s.set_source_slots(np.arange(B))
            s.set_receiver_slots(np.arange(4 * B) % B)
            s.prepare_fields(prec, 9 if prec in (N.F16, N.BF16) else 0)
            s.run(sc.n_steps, prec)
            raw = {N.F32: np.float32, N.F64: np.float64, N.F16: np.float16, N.BF16: np.uint16}[prec]
            out.append((s.responses(), *s.fields_raw(raw)))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
