"""The pass-1 work list of many billboards with a large radius among them: depth
slices make it longer, which must not make a call fail that fits without them.
The occupancy is the oracle's."""
from dataclasses import replace

import numpy as np
import pytest

import oracle_lib as O
from gpu_common import log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [96, 64])
@pytest.mark.parametrize("outside", [False, True])
def test_many_billboards(cv, gpu_ctx, N, outside):
    """One large billboard among small ones, and (outside) as many large ones
    that leave no pixel on the light image."""
    S, big = 400_000, 20.0
    log(f"[work list] N={N} S={S} outside={outside}")
    rng = np.random.default_rng(N)
    xyz = rng.uniform(-0.9, 0.9, size=(S, 3)).astype(np.float32)
    r = np.full(S, 0.2 / N, np.float32)
    if outside:
        sun = np.array([0.0, 0.0, 1.0])
        xyz[40:, :2] = np.sign(xyz[40:, :2]) * np.float32(3.0 * big)
        r[40:] = big
    else:
        sun = np.array([0.36, 0.48, 0.8])
    r[7] = big
    xyz[7] = (0.3, -0.2, 0.1)
    base = cv.scenes.small32(1)
    sc = replace(base, N=N, levels=cv.scenes.full_levels(N), xyz=xyz, scales=r, sun_dir=sun, W=16, H=16, light_w=512,
                 light_h=509)
    want = O.voxelize(sc).state()
    assert want.any()
    vol, sun_, _, vox, _ = cv.scene_objects(sc, 0, context=gpu_ctx)
    try:
        vox.voxelize(vol, sun_)
        assert np.array_equal(vol.read_occupancy(), want)
        # a later, ordinary frame of the same volume
        vol.set_billboards(xyz[:40], np.full(40, 0.15, np.float32))
        vox.voxelize(vol, sun_)
        small = O.voxelize(replace(sc, xyz=xyz[:40], scales=np.full(40, 0.15, np.float32))).state()
        assert np.array_equal(vol.read_occupancy(), small)
    finally:
        vol.close()
