"""Frames at the sizes where their launches change: the work list, the camera
setup with the sort, and the tile order made by one workgroup (1024 billboards,
4096 tiles at most) and by several; billboards of one pass-1 tile, of a few and
of more than a wave's 64; sorted and upload order.  Occupancy and image are the
oracle's bit for bit."""
from dataclasses import replace

import numpy as np
import pytest

from gpu_common import assert_bit_equal, log, run_gpu, run_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,W,H,light", [(1, 8, 8, 64), (2, 512, 512, 640), (255, 513, 512, 320), (257, 96, 64, 1400),
                                         (1024, 200, 120, 256), (1025, 200, 120, 256)])
@pytest.mark.parametrize("fmt", [1, 2])
def test_frame(cv, gpu_ctx, S, W, H, light, fmt):
    log(f"[launches] S={S} {W}x{H} light={light} fmt={fmt}")
    base = cv.scenes.small32(S)
    rng = np.random.default_rng(S + light)
    xyz = rng.uniform(-0.7, 0.7, size=(S, 3)).astype(np.float32)
    r = rng.uniform(0.01, 0.08, size=S).astype(np.float32)
    r[:: max(S // 3, 1)] = rng.uniform(0.2, 0.9, size=r[:: max(S // 3, 1)].size)
    sc = replace(base, xyz=xyz, scales=r, W=W, H=H, light_w=light, light_h=light - 9, fmt=fmt,
                 cone=replace(base.cone, steps=12))
    o = run_oracle(sc, want_f64=False)
    g = run_gpu(cv, sc, ctx=gpu_ctx, read_levels=False)
    assert np.array_equal(g.state, o.vox.state())
    assert_bit_equal("image", g.image, o.img32)
