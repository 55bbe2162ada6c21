"""The converged reference at the edges of its rounds (k_ground_truth: four
waves of 8 samples, at most 64 samples a launch) and of its 8x8 tiles: sums
bit-exact against the oracle, as in test_gpu_ground_truth."""
import numpy as np
import pytest

import oracle as O
from _parity import params_for_oracle
from smallproject_amd import configs
from test_gpu_ground_truth import _oracle_gt, _xorshift_n

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size,spp", [((61, 37), 1), ((61, 37), 7), ((40, 24), 9), ((61, 37), 31), ((33, 41), 33),
                                      ((61, 37), 65)])
def test_rounds(gpu, size, spp):
    sc = configs.CONFIGS["c2_area_1024"]
    W, H = size
    w = configs.build_world(sc, W, H)
    w.force_sync()
    w.look_at(*sc.camera(sc.frames // 2))
    p = w.prepare_frame()
    got = w.renderer.ground_truth(p, spp, frame0=5).reshape(-1)
    ocfg = O.make_config(W, H, sc.point, gfxexp=1, quirks=sc.quirks, lut=np.array(list(w.cfg.emit_lut), np.float32))
    view, op = O.View(w.grid(), w.bricks()), params_for_oracle(p)
    want = None
    for done in range(0, spp, 64):
        q = O.Params.from_buffer_copy(bytes(op))
        q.R0 = _xorshift_n(op.R0, done)
        want = _oracle_gt(ocfg, q, view, min(64, spp - done), 5 + done, want)
    w.close()
    assert np.count_nonzero(want) > 0
    same = got.view(np.uint64) == want.view(np.uint64)
    assert same.all(), f"{size} {spp} spp: {int((~same).sum())} of {same.size} sums differ"
