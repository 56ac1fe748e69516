"""Rooms that the large tile of the several-level sweep takes whatever the cost model says: their four
fields exceed 256 MB. One to three tiles along x and y, a little more or less, and many slices."""
import numpy as np

from parallelfdtd_amd import native as N
from parallelfdtd_amd import rooms

ELEM = {N.F32: 4, N.F64: 8, N.F16: 2, N.BF16: 2, N.F16_DIFF: 2}
# owned columns and rows of a block, halo columns, most levels
TILE = {p: (56, 56, 4, 4) if p == N.F64 else (112, 38, 8, 5) for p in ELEM}
# columns and rows beside whole tiles, z-chunk, steps
BORDERS = [(-2, 1, 0, 23), (0, 0, 3, 9), (2, -1, 5, 14), (1, 5, 0, 7), (9, 6, 64, 11)]


def dims(prec, dx, dy):
    ox, oy, _, _ = TILE[prec]
    X, Y = 2 * ox + dx, 2 * oy + dy
    if prec == N.F16_DIFF:
        X += X % 2
    return X, Y, (256 << 20) // (4 * ELEM[prec] * X * Y) + 3


def scene(prec, dx, dy, n_steps, centred=False, seed=1400):
    """Sources in the columns and rows that neighbouring tiles share, on few slices, receivers beside them;
    boxes on tile borders (forward boundaries)."""
    X, Y, Z = dims(prec, dx, dy)
    ox, oy, hx, lm = TILE[prec]
    sc = rooms.scene_random_small(seed + dx, dims=(X, Y, Z), n_mat=4, n_boxes=0, n_src=10, n_rec=80, n_steps=n_steps)
    rng = np.random.default_rng(seed + dy)
    if not centred:
        for z in (6, Z // 2 + 5, Z - 12):
            sc.labels[z:z + 4, oy - 3:oy + 2, ox - 2:ox + 6] = 2
            sc.labels[z:z + 6, 3:Y - 3, ox // 2:ox // 2 + 3] = 4
    n = 10
    x = rng.choice([1, hx, ox - hx, ox - 1, ox, ox + hx - 1, X - 2], n)
    y = rng.choice([1, lm, oy - lm, oy - 1, oy, oy + lm - 1, Y - 2], n)
    z = rng.choice([2, Z // 2, Z - 4], n) + rng.integers(-1, 2, n)
    sc.src_xyz = np.clip(np.stack([x, y, z], 1), 1, np.array([X, Y, Z]) - 2).astype(np.int32)
    near = np.repeat(sc.src_xyz, 8, axis=0)
    sc.rec_xyz = np.clip(near + rng.integers(-2, 3, near.shape), 1, np.array([X, Y, Z]) - 2).astype(np.int32)
    return sc
