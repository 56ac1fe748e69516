"""The context's host code on the stand-in HIP runtime: what it holds and launches when an allocation
fails, and what it gives back."""
import numpy as np
import pytest

import hostrt
import large_tile
from parallelfdtd_amd import native as N
from parallelfdtd_amd import rooms
from parallelfdtd_amd.solver import Solver


@pytest.fixture(scope="module")
def rt(tmp_path_factory):
    r = hostrt.Runtime(hostrt.build(tmp_path_factory.mktemp("hostrt")))
    kept, N._lib = N._lib, r.lib
    yield r
    N._lib = kept


@pytest.fixture(autouse=True)
def no_limits(rt):
    yield
    rt.fail_malloc(-1)
    rt.budget(1 << 40)
    rt.log()


def scene(dims, n_src=2, n_rec=5, n_steps=12, seed=5):
    return rooms.scene_random_small(seed, dims=dims, n_mat=3, n_boxes=2, n_src=n_src, n_rec=n_rec,
                                    n_steps=n_steps)


def sweeps(rt):
    return [l for l in rt.log() if l.startswith(("sweep", "row_bits"))]


FIELDS = 4  # allocations of a run whose failure refuses it: the four fields


@pytest.mark.parametrize("first,then", [(N.F64, N.F32), (N.F32, N.F64)])
@pytest.mark.parametrize("fail", range(9))
def test_an_allocation_fails_at_a_change_of_tile(rt, first, then, fail):
    """FP32 and FP64 take other tiles: planes and events are rebuilt at the change. Whichever allocation
    fails there, the run falls back (or is refused for its fields), and every later sweep reads planes
    and events of its own tile."""
    with Solver() as s:
        s.load_scene(scene((131, 50, 17), n_rec=40))
        s.run(12, first)
        assert all(l.endswith("bad=none") for l in sweeps(rt))
        s.set_receivers(np.tile([[9, 9, 9]], (400, 1)))  # more events than there is room for so far
        rt.fail_malloc(fail)
        try:
            s.run(12, then)
            assert fail >= FIELDS
        except N.PfdtdError as e:
            assert e.code == N.E_NOMEM and fail < FIELDS + 1  # the responses after the fields
        rt.fail_malloc(-1)
        for prec in (first, then, first):
            s.run(12, prec)
            lines = sweeps(rt)
            assert lines and all(l.endswith("bad=none") for l in lines), lines


def batch(s, dims, B, prec, layout=N.BATCH_INTERLEAVED):
    s.load_scene(scene(dims, n_src=B, n_rec=B))
    s.set_batch_layout(layout)
    s.set_batch(B)
    s.set_source_slots(np.arange(B))
    s.set_receiver_slots(np.arange(B))
    s.prepare_fields(prec, 9 if prec in (N.F16, N.BF16) else 0)


@pytest.mark.parametrize("prec", [N.F32, N.F64, N.F16, N.BF16])
def test_steps_of_a_prepared_batch_take_the_interleaved_update(rt, prec):
    """One launch of the interleaved update per step, also without begin_steps, before and after a run
    that held the fields slot by slot."""
    with Solver() as s:
        batch(s, (60, 40, 20), 8, prec)
        rt.log()
        s.step(0)
        prepared = rt.log()
        s.begin_steps(12, prec)
        rt.log()
        s.step(0)
        assert rt.log()[:2] == prepared[:2] and len([l for l in prepared if "update" in l]) == 1, prepared
        s.run(12, prec)
        assert any(l.startswith("sweep") and "slots=8" in l for l in rt.log())
        s.prepare_fields(prec, 9 if prec in (N.F16, N.BF16) else 0)
        rt.log()
        s.step(0)
        assert rt.log()[:2] == prepared[:2]


@pytest.mark.parametrize("prec,es", [(N.F32, 4), (N.F16, 2)])
def test_contexts_with_batches_fit_where_two_fields_each_fit(rt, prec, es):
    """An interleaved batch does with two fields: a card with room for two such contexts, and a little
    more, holds both, whatever the first one runs. With plenty of room a run takes four."""
    dims, B = (120, 80, 40), 8
    field = es * 120 * 80 * 40 * B
    rt.budget(rt.used() + 4 * field + (5 << 20))
    with Solver() as s, Solver() as t:
        for x in (s, t):
            batch(x, dims, B, prec)
            x.run(12, prec)
            assert not any("slots=8" in l for l in rt.log())
    rt.budget(1 << 40)
    with Solver() as s:
        before = rt.used()
        batch(s, dims, B, prec)
        s.run(12, prec)
        assert rt.used() - before > 4 * field
        assert any("slots=8 bad=none" in l for l in rt.log())


def test_responses_fit_beside_the_fields_of_a_batch(rt):
    """A card with room for the two fields of an interleaved batch, its planes and its responses."""
    dims, B, steps = (60, 40, 20), 8, 40000
    field, resp = 4 * 60 * 40 * 20 * B, 8 * B * steps
    rt.budget(rt.used() + 2 * field + resp + (2 << 20))
    with Solver() as s:
        batch(s, dims, B, N.F32)
        s.run(steps, N.F32)


@pytest.mark.parametrize("prec", [N.F32, N.F64, N.F16])
def test_planes_of_a_room_are_given_back_with_it(rt, prec):
    """A context that goes on to a room of another size holds what a fresh one on that room holds, and
    fits a larger room where a fresh one fits."""
    def on(*dims):
        with Solver() as s:
            for d in dims:
                s.load_scene(scene(d))
                s.run(12, prec)
            return rt.used()

    big, small, bigger = (150, 110, 80), (40, 30, 20), (160, 112, 84)
    # what the context keeps of the larger room is no more than its few events
    assert on(big, small) <= on(small) + 4096
    held = on(bigger)
    rt.budget(held + 4096)
    on(big, bigger)


@pytest.mark.parametrize("prec,raw", [(N.F32, np.float32), (N.F16, np.float16)])
def test_fields_of_a_run_are_read_on_a_full_card(rt, prec, raw):
    """A batch's fields are read out after a run without an allocation on the card."""
    with Solver() as s:
        batch(s, (60, 40, 20), 8, prec)
        s.run(12, prec)
        assert any("slots=8 bad=none" in l for l in rt.log())
        rt.budget(rt.used())
        P, Pp = s.fields_raw(raw)
        assert P.shape == (20, 40, 60, 8)


# rooms of the large tile: whether a call of one step takes the single-step update, and of two steps
# the two-column sweep
SHORT_CALLS = [
    ((256, 256, 256), N.F32, False, True, False), ((384, 320, 256), N.F32, False, False, False),
    ((130, 98, 66), N.F32, False, False, False), ((448, 264, 135), N.F32, True, True, False),
    ((384, 320, 256), N.F64, False, False, False), ((640, 480, 320), N.F64, False, True, False),
    ((256, 256, 256), N.F16, False, True, False), ((640, 480, 320), N.F16, False, False, False),
    ((1024, 768, 384), N.F16, False, False, True), ((1023, 768, 384), N.F16, False, False, False),
    ((256, 256, 256), N.BF16, False, True, False), ((640, 480, 320), N.BF16, False, False, False),
]


@pytest.mark.parametrize("dims,prec,centred,single,pair", SHORT_CALLS)
def test_short_calls_take_the_faster_kernels(rt, dims, prec, centred, single, pair):
    lab = rooms.box_room(*dims)
    with Solver() as s:
        if centred:
            s.set_update_type(N.SRL)
        s.set_domain_labels(lab)
        s.set_materials(np.full((1, 20), 0.1, np.float32))
        s.begin_steps(20, prec)
        got = {}
        for first, n in ((0, 1), (1, 2), (3, 6), (9, 4)):
            rt.log()
            s.steps(first, n)
            got[n] = [l for l in rt.log() if "inject" not in l]
    is_sweep = lambda l: l.startswith("sweep")
    assert all("update_kernel" in l if single else is_sweep(l) and "levels=1" in l for l in got[1][-1:])
    assert all(("update2" in l) if pair else is_sweep(l) for l in got[2][-1:])
    assert is_sweep(got[4][-1])
    if not got[6][-1].startswith("sweep") or "levels=1 " in got[6][-1]:  # five levels and a single step
        assert is_sweep(got[6][-2]) and ("update_kernel" in got[6][-1]) == single


@pytest.mark.parametrize("dx,dy,zchunk,n_steps", large_tile.BORDERS)
@pytest.mark.parametrize("prec,centred", [(p, c) for p in large_tile.ELEM for c in (False, True)
                                          if not (c and p == N.F16_DIFF)])
def test_rooms_of_the_large_tile_take_it(rt, prec, centred, dx, dy, zchunk, n_steps):
    """The rooms of the GPU tests of the large tile."""
    ox, oy, hx, lm = large_tile.TILE[prec]
    with Solver() as s:
        if centred:
            s.set_update_type(N.SRL)
        s.set_time_levels(0, zchunk)
        s.set_domain_labels(rooms.box_room(*large_tile.dims(prec, dx, dy)))
        s.set_materials(np.full((1, 20), 0.1, np.float32))
        rt.log()
        s.run(n_steps, prec)
        lines = [l for l in rt.log() if l.startswith("sweep")]
    assert lines and all(f"tile={ox},{hx},{oy}," in l and l.endswith("bad=none") for l in lines), lines
    assert f"levels={min(lm, n_steps)} " in lines[0]
