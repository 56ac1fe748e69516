"""The work that users of this framework have it do, as measured cases.

Every case goes through the Python host objects over the C ABI (``Solver``, ``Pool``) the way a
program that computes room impulse responses does:

* ``run``:   one whole simulation of a voxel room (`Solver.run`) and its receiver responses;
* ``batch``: several source positions of one room in one run (both field layouts);
* ``pool``:  a set of impulse-response jobs served through one pool, from submission to
             responses;
* ``mesh``:  a triangle mesh voxelized, then stepped with slices of the field captured on the
             way (the App's geometry and capture flow), with the centred boundaries.

Rooms, obstacles, materials, sources, receivers and signals come from the seed.
"""
from __future__ import annotations

import math
import time

import numpy as np
import torch

from parallelfdtd_amd import geometry as G
from parallelfdtd_amd import native as N
from parallelfdtd_amd import rooms
from parallelfdtd_amd.rooms import LAMBDA, SplitMix64
from parallelfdtd_amd.serve import JobSpec, Pool
from parallelfdtd_amd.solver import Solver, voxel_grid

PRECISION = {"f32": N.F32, "f64": N.F64, "f16": N.F16, "bf16": N.BF16, "f16diff": N.F16_DIFF}
BYTES = {"f32": 4, "f64": 8, "f16": 2, "bf16": 2, "f16diff": 2}
SCALE_EXP = 12  # storage scale 2^12 of the 16-bit formats, for unit-peak sources
NODE_STEPS_EXACT = 1.6e11  # about 20 s of the 64-bit evaluation on this card
NODES_EXACT = 6e8  # its fields and coefficients take 48 bytes per node and as much while built
MESH_PAD = (32, 4, 1)  # the App's padding
MESH_DX = 1.0 / 32


def listed() -> list[dict]:
    return [
        # The smallest whole simulation: one source and one receiver in a 128 x 96 x 64 box of
        # air, 2000 steps. Everything fits in cache; launches and per-step latency count.
        dict(name="box_f32", kind="run", X=130, Y=98, Z=66, hall=False, boxes=0, n_mat=1,
             n_src=1, n_rec=1, steps=2000, precision="f32"),
        # A study at odd sizes in double precision: a small furnished room, several sources and
        # receivers.
        dict(name="odd_room_f64", kind="run", X=157, Y=111, Z=75, hall=False, boxes=5, n_mat=3,
             n_src=3, n_rec=12, steps=1000, precision="f64"),
        # The ordinary job: an L-shaped hall of 302 M nodes with pillars, in single and in
        # double precision.
        dict(name="hall_f32", kind="run", X=1024, Y=768, Z=384, hall=True, boxes=8, n_mat=5,
             n_src=1, n_rec=16, steps=300, precision="f32"),
        dict(name="hall_f64", kind="run", X=1024, Y=768, Z=384, hall=True, boxes=8, n_mat=5,
             n_src=1, n_rec=16, steps=150, precision="f64"),
        # The largest room: 2.4 G nodes (past 2^31), in single precision and with 16-bit fields.
        dict(name="large_f32", kind="run", X=2048, Y=1536, Z=768, hall=False, boxes=32, n_mat=8,
             n_src=1, n_rec=64, steps=120, precision="f32"),
        dict(name="large_f16", kind="run", X=2048, Y=1536, Z=768, hall=False, boxes=32, n_mat=8,
             n_src=1, n_rec=64, steps=120, precision="f16"),
        # 16-bit fields on a room whose sizes come from its geometry: odd and ragged.
        dict(name="ragged_bf16", kind="run", X=701, Y=523, Z=307, hall=False, boxes=10, n_mat=6,
             n_src=2, n_rec=16, steps=400, precision="bf16"),
        # The difference form, for the smallest in-band error with 16-bit fields.
        dict(name="hall_f16diff", kind="run", X=640, Y=480, Z=320, hall=True, boxes=6, n_mat=5,
             n_src=1, n_rec=16, steps=400, precision="f16diff"),
        # Many source positions in one furnished room of 50 M nodes: the layout that the
        # autotuner chooses (8 sources), and the default layout with 32.
        dict(name="sources8_grouped", kind="batch", X=512, Y=384, Z=256, boxes=12, n_mat=4,
             slots=8, grouped=True, rec_per_slot=8, steps=150, precision="f32"),
        dict(name="sources32_interleaved", kind="batch", X=512, Y=384, Z=256, boxes=12, n_mat=4,
             slots=32, grouped=False, rec_per_slot=8, steps=60, precision="f32"),
        # Serving: sixteen jobs of rooms of 64..384 per side, both storage types, through one
        # pool, from submission to responses.
        dict(name="serve16", kind="pool", jobs=16, side_min=64, side_max=384, steps_min=300,
             steps_max=900),
        # A triangle mesh at 1/32 m, centred boundaries, a horizontal slice every 25 steps.
        dict(name="mesh_capture", kind="mesh", X=420, Y=261, Z=133, obstacles=4, n_rec=8,
             steps=300, every=25, precision="f32"),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.499)))))


def draw(rng) -> dict:
    kind = rng.choice(["run"] * 6 + ["batch"] * 2 + ["pool", "mesh"])
    if kind == "pool":
        lo = _log_int(rng, 48, 160)
        smin = rng.randint(100, 600)
        return dict(kind=kind, jobs=rng.randint(2, 16), side_min=lo,
                    side_max=lo + rng.randint(16, 200), steps_min=smin,
                    steps_max=smin + rng.randint(0, 400))
    if kind == "mesh":
        steps = rng.randint(60, 400)
        return dict(kind=kind, X=_log_int(rng, 90, 640), Y=_log_int(rng, 60, 400),
                    Z=_log_int(rng, 40, 200), obstacles=rng.randint(0, 5),
                    n_rec=rng.randint(1, 16), steps=steps, every=rng.randint(10, 50),
                    precision=rng.choice(["f32", "f32", "f64", "f16"]))
    if kind == "batch":
        X = _log_int(rng, 96, 512)
        Y, Z = int(X * rng.uniform(0.5, 1.0)), int(X * rng.uniform(0.3, 0.8))
        slots = rng.choice([2, 4, 8, 16, 32])
        steps = int(max(30, min(400, rng.uniform(0.3, 1.0) * 8e10 / (X * Y * Z * slots))))
        return dict(kind=kind, X=X, Y=Y, Z=Z, boxes=rng.randint(0, 12), n_mat=rng.randint(1, 6),
                    slots=slots, grouped=rng.random() < 0.5, rec_per_slot=rng.randint(1, 8),
                    steps=steps, precision=rng.choice(["f32", "f32", "f64", "f16"]))
    X = _log_int(rng, 64, 2048)
    Y = min(1536, int(X * rng.uniform(0.4, 1.1)) + 8)
    Z = min(768, int(X * rng.uniform(0.25, 0.9)) + 8)
    precision = rng.choice(["f32", "f32", "f64", "f16", "bf16", "f16diff"])
    most = 8e8 if precision == "f64" else 2.4e9  # states are held several times over
    Z = max(8, min(Z, int(most / (X * Y))))
    if precision == "f16diff":
        X += X % 2  # the difference form takes rooms of even width
    budget = rng.uniform(0.2, 1.0) * 7e10 * (0.5 if precision == "f64" else 1.0)
    steps = int(max(30, min(2000, budget / (X * Y * Z))))
    return dict(kind="run", X=X, Y=Y, Z=Z, hall=rng.random() < 0.4, boxes=rng.randint(0, 16),
                n_mat=rng.randint(5, 8), n_src=rng.choice([1, 1, 2, 4]),
                n_rec=rng.randint(1, 64), steps=steps, precision=precision)


# ---- inputs --------------------------------------------------------------------------------

def _near(lab, rng: SplitMix64, src, n: int, reach: int) -> np.ndarray:
    """n air points within `reach` voxels of a source: listeners that hear it within the run."""
    Z, Y, X = lab.shape
    pts = []
    for k in range(n):
        s = src[k % len(src)]
        r = reach
        for t in range(2000):
            x, y, z = (int(s[a]) + rng.randint(-r, r) for a in range(3))
            if rooms.is_air_k6(lab, x, y, z):
                pts.append((x, y, z))
                break
            r = max(1, r - (t % 50 == 49))
        else:
            pts.append(tuple(int(v) for v in s))
    return np.asarray(pts, np.int32).reshape(n, 3)


def _receivers(lab, rng: SplitMix64, src, n: int, steps: int) -> np.ndarray:
    """Half of the receivers near the sources, half anywhere in the room."""
    near = (n + 1) // 2
    pts = _near(lab, rng, src, near, max(3, steps // 5))
    return np.concatenate([pts, rooms.seeded_points(lab, rng, n - near)]).astype(np.int32)


def _signals(rng: SplitMix64, n: int, steps: int) -> np.ndarray:
    """Unit-scale pulses: Gaussians and band-limited Gaussian derivatives, one per source."""
    out = []
    for k in range(n):
        sigma = rng.uniform(5.0, 12.0)
        pulse = rooms.gaussian_pulse if k % 2 else rooms.gaussian_derivative_pulse
        out.append(rng.uniform(0.5, 1.0) * pulse(steps, 5.0 * sigma, sigma))
    return np.asarray(out).reshape(n, steps)


def _room(case: dict, seed: int):
    """(labels, admittances, rng) of a box room or an L-shaped hall with solid boxes in it."""
    rng = SplitMix64(seed)
    X, Y, Z, m = case["X"], case["Y"], case["Z"], case["n_mat"]
    betas = np.array([rng.uniform(0.01, 0.6) for _ in range(m)], np.float32)
    lab = rooms.box_room(X, Y, Z, floor=0, ceiling=min(1, m - 1), walls=min(2, m - 1))
    if case.get("hall"):
        x0, y0 = int(X * rng.uniform(0.4, 0.7)), int(Y * rng.uniform(0.4, 0.7))
        lab[1:Z - 1, y0:, x0:] = min(3, m - 1) + 1
    smax = max(3, min(X, Y, Z) // 4)
    rooms.add_boxes(lab, rng.fork(3), case["boxes"], max(2, smax // 8), smax,
                    list(range(min(3, m - 1), m)))
    return lab, betas, rng


def _table(betas) -> np.ndarray:
    return np.repeat(betas.astype(np.float32)[:, None], 20, axis=1)


def _run_inputs(case, seed):
    lab, betas, rng = _room(case, seed)
    src = rooms.seeded_points(lab, rng.fork(4), case["n_src"])
    rec = _receivers(lab, rng.fork(5), src, case["n_rec"], case["steps"])
    return lab, betas, src, rec, _signals(rng.fork(6), case["n_src"], case["steps"])


def _batch_inputs(case, seed):
    lab, betas, rng = _room(case, seed)
    B, R = case["slots"], case["rec_per_slot"]
    src = rooms.seeded_points(lab, rng.fork(4), B)
    rec = np.concatenate([_receivers(lab, rng.fork(50 + b), src[b:b + 1], R, case["steps"])
                          for b in range(B)])
    return lab, betas, src, rec, _signals(rng.fork(6), B, case["steps"])


def _pool_specs(case, seed) -> list[JobSpec]:
    out = []
    for j in range(case["jobs"]):
        rng = SplitMix64(seed).fork(100 + j)
        # the sides of the jobs spread over the whole range, whatever the seed
        X, Y, Z = (case["side_min"] + (case["side_max"] - case["side_min"]) *
                   ((j * q + rng.randint(0, 3)) % 16) // 15 for q in (5, 7, 3))
        steps = case["steps_min"] + (case["steps_max"] - case["steps_min"]) * ((j * 11) % 16) // 15
        m = 1 + j % 6
        lab, betas, rng = _room(dict(X=X, Y=Y, Z=Z, n_mat=m, boxes=j % 11), rng.next_u64())
        src = rooms.seeded_points(lab, rng.fork(4), 1 + (j * 7) % 16)
        rec = _receivers(lab, rng.fork(5), src, 4, steps)
        sig = _signals(rng.fork(6), len(src), min(steps, 200))
        half = j % 2 == 1
        out.append(JobSpec(lab, betas, src, np.ones(len(src), np.int32), sig.astype(np.float32),
                           rec, steps, N.F16 if half else N.F32, SCALE_EXP if half else 0))
    return out


def _mesh_boxes(case, seed):
    """Obstacles of the mesh room, in nodes: one per strip of its length, apart from each other
    and from the walls, with faces between the node planes."""
    rng = SplitMix64(seed).fork(7)
    X, Y, Z, n = case["X"], case["Y"], case["Z"], case["obstacles"]
    out = []
    for k in range(n):
        lo, hi = X * k // n + 4, X * (k + 1) // n - 4
        x0 = rng.randint(lo, max(lo, (lo + hi) // 2 - 2))
        x1 = rng.randint(x0 + 2, max(x0 + 2, hi))
        y0 = rng.randint(4, Y // 2 - 3)
        y1 = rng.randint(y0 + 2, Y - 4)
        z0 = rng.randint(4, Z // 2 - 3)
        z1 = rng.randint(z0 + 2, Z - 4)
        out.append(tuple(v + 0.5 for v in (x0, y0, z0, x1, y1, z1)))
    return out


def _mesh_inputs(case, seed):
    """Triangles of a box room (a material per face) with box obstacles (a material each)."""
    room = G.box_mesh((0, 0, 0), tuple((case[a] - 0.5) * MESH_DX for a in "XYZ"))
    names = list(room.layers)
    verts, tris = [room.vertices], [room.indices]
    mats = [G.layer_materials(room, {n: k for k, n in enumerate(names)})]
    boxes = _mesh_boxes(case, seed)
    for k, b in enumerate(boxes):
        m = G.box_mesh(tuple(v * MESH_DX for v in b[:3]), tuple(v * MESH_DX for v in b[3:]))
        tris.append(m.indices + sum(len(v) for v in verts))
        verts.append(m.vertices)
        mats.append(np.full(len(m.indices), 6 + k, np.uint8))
    rng = SplitMix64(seed).fork(8)
    betas = np.array([rng.uniform(0.01, 0.6) for _ in range(6 + len(boxes))], np.float32)

    def free(p):  # clear of the walls and obstacles
        return not any(all(b[a] - 2 <= p[a] - 1 <= b[a + 3] + 2 for a in range(3)) for b in boxes)

    def point(lo, hi):
        while True:
            p = tuple(rng.randint(max(3, lo[a]), min(case["XYZ"[a]] - 3, hi[a])) for a in range(3))
            if free(p):
                return p

    src = point((0, 0, 0), (10 ** 6,) * 3)
    rec, reach = [], max(6, case["steps"] // 5)
    for k in range(case["n_rec"]):
        r = reach if k % 2 == 0 else 10 ** 6
        rec.append(point([v - r for v in src], [v + r for v in src]))
    return (np.concatenate(verts).astype(np.float32), np.concatenate(tris).astype(np.uint32),
            np.concatenate(mats).astype(np.uint8), names, boxes, betas,
            np.array([src], np.int32), np.array(rec, np.int32),
            _signals(rng.fork(6), 1, case["steps"]))


# ---- the cases as a user's program runs them -------------------------------------------------

def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind == "pool":
        specs = _pool_specs(case, seed)
        need = sum(Pool.job_bytes(s) for s in specs)
        return {"case": case, "pool": Pool(0, need + need // 4 + (64 << 20)), "specs": specs}
    s = Solver(0)
    if kind == "mesh":
        v, t, m, _names, _boxes, betas, src, rec, sig = _mesh_inputs(case, seed)
        s.set_update_type(N.SRL)
        st = {"case": case, "solver": s, "vertices": v, "triangles": t, "materials": m,
              "dims": voxel_grid(v, MESH_DX, MESH_PAD)}
    else:
        inputs = _batch_inputs if kind == "batch" else _run_inputs
        lab, betas, src, rec, sig = inputs(case, seed)
        s.set_domain_labels(lab)
        st = {"case": case, "solver": s}
    s.set_materials(_table(betas))
    if kind == "batch":
        s.set_batch_layout(N.BATCH_GROUPED if case["grouped"] else N.BATCH_INTERLEAVED)
        s.set_batch(case["slots"])
    s.set_sources(src, np.ones(len(src), np.int32), signal_f64=sig,
                  signal_f32=sig.astype(np.float32))
    s.set_receivers(rec)
    if kind == "batch":
        s.set_source_slots(np.arange(case["slots"]))
        s.set_receiver_slots(np.repeat(np.arange(case["slots"]), case["rec_per_slot"]))
    if kind != "mesh":
        p = case["precision"]
        s.prepare_fields(PRECISION[p], SCALE_EXP if BYTES[p] == 2 else 0)
    return st


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "pool":
        return _serve(state["pool"], state["specs"])
    s = state["solver"]
    p = PRECISION[case["precision"]]
    if kind != "mesh":
        s.run(case["steps"], p)
        return s.responses()
    s.voxelize(state["vertices"], state["triangles"], MESH_DX, state["materials"], MESH_PAD)
    if BYTES[case["precision"]] == 2:
        s.prepare_fields(p, SCALE_EXP)
    s.begin_steps(case["steps"], p)
    slices, k = [], 0
    while k < case["steps"]:
        n = min(case["every"], case["steps"] - k)
        s.steps(k, n)
        k += n
        slices.append(s.capture_slice(state["dims"][2] // 2, 0))
    return {"responses": s.responses(), "pressure": np.stack([a for a, _ in slices]),
            "position": np.stack([b for _, b in slices])}


def _serve(pool: Pool, specs) -> list:
    """All jobs submitted, bundles kept flowing, every finished job's responses collected."""
    ids = [pool.submit(s) for s in specs]
    got, active = {}, 1
    while len(got) < len(ids):
        active = pool.advance()
        for j in pool.poll():
            got[j] = pool.responses(j)
            pool.release(j)
        if active == 0:
            time.sleep(2e-4)
    return [got[j] for j in ids]


# ---- work ------------------------------------------------------------------------------------

def _rooms_of(case):
    """[(nodes, steps, copies of the fields, storage bytes, receivers)] of the case's rooms."""
    kind = case["kind"]
    if kind == "pool":
        out = []
        for s in _pool_shapes(case):
            out.append((s[0], s[1], 1, s[2], 4))
        return out
    n = case["X"] * case["Y"] * case["Z"]
    if kind == "mesh":
        n = math.prod(-(-(case[a] + 2) // q) * q for a, q in zip("XYZ", MESH_PAD))
    b = case.get("slots", 1)
    rec = case["n_rec"] if kind != "batch" else b * case["rec_per_slot"]
    return [(n, case["steps"], b, BYTES[case["precision"]], rec)]


def _pool_shapes(case):
    """(nodes, steps, storage bytes) per job, sides at the middle of the seeds' spread."""
    span, lo = case["side_max"] - case["side_min"], case["side_min"]
    for j in range(case["jobs"]):
        n = math.prod(lo + span * ((j * q + 1) % 16) // 15 for q in (5, 7, 3))
        steps = case["steps_min"] + (case["steps_max"] - case["steps_min"]) * ((j * 11) % 16) // 15
        yield n, steps, 2 if j % 2 else 4


def work(case: dict) -> dict:
    """Bytes: the room's position and material bytes read once and the two fields of the last
    step written once, the responses and captured slices written. Operations: five additions,
    four products, an addition and a subtraction per node and step."""
    nbytes = flops = 0
    for n, steps, copies, size, rec in _rooms_of(case):
        nbytes += n * (2 + 2 * size * copies) + 8 * rec * steps
        flops += 11 * n * steps * copies
    if case["kind"] == "mesh":
        plane = math.prod(-(-(case[a] + 2) // q) * q for a, q in zip("XY", MESH_PAD))
        nbytes += 5 * plane * -(-case["steps"] // case["every"])
    return {"bytes": nbytes, "flops": flops}


# ---- 64-bit results --------------------------------------------------------------------------

SHIFTS = [(2, -1), (2, 1), (1, -1), (1, 1), (0, -1), (0, 1)]  # -x +x -y +y -z +z


def _nb(t, axis, d):
    """The interior's neighbours along one axis of a (Z, Y, X) tensor."""
    sl = [slice(1, -1)] * 3
    sl[axis] = slice(0, -2) if d < 0 else slice(2, None)
    return t[tuple(sl)]


class _Exact:
    """The update rule in 64 bits with torch operations, on a label grid."""

    def __init__(self, lab, betas, centred=False):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        lab = torch.from_numpy(np.ascontiguousarray(lab)).to(dev)
        self.shape, self.dev = lab.shape, dev
        f64 = torch.float64
        inside = lab == 0
        mid = inside[1:-1, 1:-1, 1:-1]
        K = torch.zeros(mid.shape, dtype=f64, device=dev)
        mat = torch.zeros(mid.shape, dtype=torch.uint8, device=dev)
        for axis, d in reversed(SHIFTS):
            air = _nb(inside, axis, d)
            K += air
            mat = torch.where(air, mat, _nb(lab, axis, d) - 1)
        b = torch.zeros(256, dtype=f64, device=dev)
        b[:len(betas)] = torch.from_numpy(betas.astype(np.float64)).to(dev)
        lam2 = LAMBDA * LAMBDA
        self.mirror = None
        if centred:
            # a missing neighbour is replaced by the present one across the node
            self.mirror = [1.0 + (~_nb(inside, axis, -d)).to(f64) for axis, d in SHIFTS]
            beta = b[mat.long()] * LAMBDA * (6.0 - K)
            self.a = torch.full_like(K, -(2.0 - 6.0 * lam2))
        else:
            beta = 0.5 * b[mat.long()] * (6.0 - K) * LAMBDA
            self.a = 2.0 - K * lam2
        g = mid.to(f64) / (1.0 + beta)
        self.a *= g
        self.c = g * (1.0 - beta)
        self.s = g * lam2

    def run(self, src, sig, rec, steps, capture=None):
        """Responses [n_rec][steps]; capture = (slice, every): also the slices taken."""
        P = torch.zeros(self.shape, dtype=torch.float64, device=self.dev)
        Q = torch.zeros_like(P)
        S = torch.empty_like(self.a)
        src = torch.from_numpy(np.asarray(src, np.int64)).to(self.dev)
        rec = torch.from_numpy(np.asarray(rec, np.int64)).to(self.dev)
        sig = torch.from_numpy(np.asarray(sig, np.float64)).to(self.dev)
        out = torch.zeros((len(rec), steps), dtype=torch.float64, device=self.dev)
        inner = (slice(1, -1),) * 3
        taken = []
        for n in range(steps):
            if n < sig.shape[1]:
                P[src[:, 2], src[:, 1], src[:, 0]] += sig[:, n]
            S.zero_()
            for k, (axis, d) in enumerate(SHIFTS):
                nb = _nb(P, axis, d)
                S += nb if self.mirror is None else nb * self.mirror[k]
            S *= self.s
            q = Q[inner]
            q *= -1.0
            q *= self.c
            q += S
            q += torch.mul(self.a, P[inner], out=S)
            P, Q = Q, P
            out[:, n] = P[rec[:, 2], rec[:, 1], rec[:, 0]]
            if capture and ((n + 1) % capture[1] == 0 or n + 1 == steps):
                taken.append(P[capture[0]].cpu())
        return out.cpu().numpy(), taken


def _mesh_labels(case, seed):
    """The label grid of the mesh room in closed form: nodes at whole multiples of the edge, a
    box takes the nodes in [lo, hi), a solid node the material of the face across its first air
    neighbour."""
    _v, _t, _m, names, boxes, *_ = _mesh_inputs(case, seed)
    X, Y, Z = (-(-(case[a] + 2) // q) * q for a, q in zip("XYZ", MESH_PAD))
    air = np.zeros((Z, Y, X), bool)
    air[1:case["Z"] + 1, 1:case["Y"] + 1, 1:case["X"] + 1] = True
    lab = np.ones((Z, Y, X), np.uint8)
    n = {a: case[a] for a in "XYZ"}
    face = {f: names.index(f) + 1 for f in names}
    for first, (zs, ys, xs) in (("-z", (n["Z"] + 1, None, None)), ("+z", (0, None, None)),
                                ("-y", (None, n["Y"] + 1, None)), ("+y", (None, 0, None)),
                                ("-x", (None, None, n["X"] + 1)), ("+x", (None, None, 0))):
        wall = {"-": "+", "+": "-"}[first[0]] + first[1]
        idx = tuple(slice(None) if v is None else v for v in (zs, ys, xs))
        lab[idx] = face[wall]
    lab[air] = 0
    for k, b in enumerate(boxes):
        x0, y0, z0, x1, y1, z1 = (int(math.ceil(v)) + 1 for v in b)
        lab[z0:z1, y0:y1, x0:x1] = 7 + k
    return lab


def exact(case: dict, seed: int):
    shapes = _rooms_of(case)
    if (sum(n * s * c for n, s, c, _b, _r in shapes) > NODE_STEPS_EXACT or
            max(n for n, *_ in shapes) > NODES_EXACT):
        return None
    kind = case["kind"]
    if kind == "pool":
        out = []
        for s in _pool_specs(case, seed):
            out.append(_Exact(s.labels, s.betas).run(s.src_xyz, s.signals, s.rec_xyz, s.n_steps)[0])
        return out
    if kind == "mesh":
        *_, names, boxes, betas, src, rec, sig = _mesh_inputs(case, seed)
        lab = _mesh_labels(case, seed)
        resp, taken = _Exact(lab, betas, centred=True).run(
            src, sig, rec, case["steps"], (lab.shape[0] // 2, case["every"]))
        return {"responses": resp, "pressure": torch.stack(taken).numpy(), "position": None}
    if kind == "batch":
        lab, betas, src, rec, sig = _batch_inputs(case, seed)
        e, R = _Exact(lab, betas), case["rec_per_slot"]
        return np.concatenate([e.run(src[b:b + 1], sig[b:b + 1], rec[b * R:(b + 1) * R],
                                     case["steps"])[0] for b in range(case["slots"])])
    lab, betas, src, rec, sig = _run_inputs(case, seed)
    return _Exact(lab, betas).run(src, sig, rec, case["steps"])[0]
