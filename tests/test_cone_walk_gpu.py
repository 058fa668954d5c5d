"""The cone trace's walk over a tile's billboards at the sizes where its parts
change: candidate rounds of 64, mask words of 64 ranks and loads of 64 words,
whole and cut tiles, pixels sharing the wave's lanes.  Images and counters are
those of the oracle's FP32 pass bit for bit, whatever the split."""
from dataclasses import replace

import numpy as np
import pytest

from gpu_common import assert_bit_equal, log, run_gpu, run_oracle

pytestmark = pytest.mark.gpu


def _scene(cv, S, W, H, composite, cone_mode, fmt, march=False):
    base = cv.scenes.small32(S)
    rng = np.random.default_rng(S)
    # most billboards in one corner of the view (tiles with hundreds of
    # candidates beside empty ones), a few tiny, a few outside the view
    xyz = (rng.normal(0.0, 0.12, size=(S, 3)) + np.array([0.3, 0.2, 0.0])).astype(np.float32)
    xyz[::7] = rng.uniform(-2.0, 2.0, size=xyz[::7].shape)
    r = rng.uniform(0.02, 0.09, size=S).astype(np.float32)
    r[::11] = 0.002
    cone = replace(base.cone, steps=24, composite=composite, cone_mode=cone_mode,
                   quantize_rgba8=1 if composite == 0 else 0)
    sc = replace(base, N=32, xyz=xyz, scales=r, W=W, H=H, light_w=64, light_h=64, cone=cone, fmt=fmt)
    if cone_mode == 0:
        sc = replace(cv.scenes.reference_mode(sc), cone=replace(sc.cone, down_scaling=16.0))
    if march:
        sc = replace(sc, noise_march=cv.scenes.NoiseMarch(seed=5))
    return sc


# (billboards, width, height): candidate and word edges on small images (every
# tile in quarters), an image of more than 8192 tiles (halves), odd edges
SIZES = [(1, 9, 9), (63, 40, 24), (64, 40, 24), (65, 40, 24), (129, 97, 61), (4096, 64, 48), (4097, 64, 48),
         (300, 1000, 540)]


@pytest.mark.parametrize("S,W,H", SIZES)
@pytest.mark.parametrize("composite,cone_mode,fmt", [(1, 2, 1), (1, 1, 2), (0, 2, 2), (0, 0, 0)])
def test_walk(cv, gpu_ctx, S, W, H, composite, cone_mode, fmt):
    scene = _scene(cv, S, W, H, composite, cone_mode, fmt)
    log(f"[walk] S={S} {W}x{H} composite={composite} cone={cone_mode} fmt={fmt}")
    o = run_oracle(scene, want_f64=False)
    g = run_gpu(cv, scene, ctx=gpu_ctx, read_levels=False)
    assert_bit_equal("image", g.image, o.img32)
    gpu_ctx.set_profiling(1)
    try:
        c = run_gpu(cv, scene, ctx=gpu_ctx, read_levels=False)
    finally:
        gpu_ctx.set_profiling(0)
    assert_bit_equal("image of a counter run", c.image, o.img32)
    got = tuple(int(c.stats[k]) for k in ("fragments", "samples", "two_level"))
    assert got == (int(o.stats.fragments), int(o.stats.samples), int(o.stats.two_level))


@pytest.mark.parametrize("S", [65, 200])
def test_walk_noise_march(cv, gpu_ctx, S):
    scene = _scene(cv, S, 120, 80, 0, 0, 0, march=True)
    log(f"[walk] noise march S={S}")
    o = run_oracle(scene, want_f64=False)
    g = run_gpu(cv, scene, ctx=gpu_ctx, read_levels=False)
    assert_bit_equal("image", g.image, o.img32)
