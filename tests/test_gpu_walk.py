"""The unified walk (Walk, csrc/vr_device.h) where its bricks are left out:
bricks that hold one to three voxels, so most rays that enter one pass its
voxels by, and rays that run along voxel and brick faces, edges and
diagonals.  Every voxel, side and distance equals the oracle's bit for bit
(the same operations in the same order, so there is no tolerance)."""
import numpy as np
import pytest

import oracle as O
from smallproject_amd import World, _lib, default_config

pytestmark = pytest.mark.gpu

SIZE = 96  # voxels: 12 bricks an axis, at the map's corner and across it


def _sparse_world(base):
    w = World(default_config(64, 64, capacity=1 << 13))
    rng = np.random.default_rng(base + 1)
    cells = np.stack(np.meshgrid(*[np.arange(SIZE // 8)] * 3, indexing="ij"), -1).reshape(-1, 3)
    cells = cells[rng.random(len(cells)) < 0.6]
    # one voxel per brick at its corners, edges and inside, some with more
    for n in (1, 1, 2):
        at = rng.choice([0, 0, 3, 4, 7, 7], size=(len(cells), 3))
        keep = rng.random(len(cells)) < 1.0 / n
        xyz = base + 8 * cells[keep] + at[keep]
        words = np.where(rng.random(len(xyz)) < 0.8, 0xF000, 0x7000) | rng.integers(1, 0x1000, len(xyz))
        w.set_many(xyz.astype(np.uint32), words.astype(np.uint32))
    return w


def _rays(base, rng, n):
    lo, hi = float(base), float(base + SIZE)
    o = rng.uniform(lo, hi, (n, 3))
    o[n // 4:] = np.round(o[n // 4:] * 2) / 2          # on voxel faces and centres
    o[n // 2:n // 2 + n // 8] = np.round(o[n // 2:n // 2 + n // 8] / 8) * 8  # on brick faces
    d = rng.normal(size=(n, 3))
    d[::3] = rng.choice([-1.0, 0.0, 1.0], size=d[::3].shape)  # axes and diagonals
    d[1::5] *= rng.choice([1e-4, 1.0, 1e3], size=(len(d[1::5]), 1))
    d[(d == 0).all(1)] = (0.0, 1.0, 0.0)
    o[::2] += rng.choice([0.0, 1e-4, -1e-4], size=o[::2].shape)
    return o.astype(np.float32), d.astype(np.float32)


def _check(w, o, d, what):
    view = O.View(w.grid(), w.bricks())
    for kind in (_lib.TRACE_ALL, _lib.TRACE_OPAQUE):
        for steps in (999999, 128, 17, 5):
            gv, gd, gs = w.renderer.trace(o, d, kind, steps)
            ov, od, os_ = O.trace_batch(view, o, d, steps, kind)
            hit = ov != 0
            assert np.array_equal(gv, ov), f"{what} kind {kind} steps {steps}: {(gv != ov).sum()} voxels differ"
            assert np.array_equal(gs[hit], os_[hit]), f"{what} kind {kind} steps {steps}: side"
            assert np.array_equal(gd[hit].view(np.uint32), od[hit].view(np.uint32)), f"{what} kind {kind} steps {steps}: distance"


@pytest.mark.parametrize("base", [0, 472, 1024 - SIZE])
def test_rays_past_sparse_bricks(gpu, base):
    w = _sparse_world(base)
    w.force_sync()
    rng = np.random.default_rng(base)
    for n in (1, 63, 65, 40000):
        o, d = _rays(base, rng, n)
        _check(w, o, d, f"base {base}, {n} rays")
    # the slabs of a brick that an upload empties, fills and thins out
    full = np.stack(np.meshgrid(*[np.arange(8)] * 3, indexing="ij"), -1).reshape(-1, 3) + base + 16
    w.set_many(full.astype(np.uint32), np.full(len(full), 0xF123, np.uint32))
    w.commit()
    _check(w, o, d, "filled brick")
    w.set_many(full[1:].astype(np.uint32), np.zeros(len(full) - 1, np.uint32))
    w.commit()
    _check(w, o, d, "thinned brick")
    w.close()
