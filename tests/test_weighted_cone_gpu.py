"""The weighted cone of R8 volumes from footprint slots, and the noise march's
two-channel map, where their arithmetic changes form: sides that are and are
not multiples of the bricks, one-texel top levels, step counts and down
scalings whose product is a power of two, not, or negative, sums that saturate
and sums that do not, amplitudes that overflow and coordinates beyond the
exact integer conversion.  All bit for bit the oracle's FP32 pass."""
from dataclasses import replace

import numpy as np
import pytest

from gpu_common import assert_bit_equal, log, run_gpu, run_oracle

pytestmark = pytest.mark.gpu


def _scene(cv, N, levels, steps, ds, angle=0.6, offset=0.0):
    base = cv.scenes.reference_mode(cv.scenes.small32(N))
    cone = replace(base.cone, steps=steps, down_scaling=ds, cone_angle=angle, lod_offset=offset, quantize_rgba8=0)
    return replace(base, N=N, levels=levels, W=72, H=40, light_w=128, light_h=128, cone=cone)


@pytest.mark.parametrize("N,levels", [(1, 1), (2, 2), (3, 1), (5, 3), (16, 5), (17, 5), (31, 4), (48, 6), (64, 7)])
@pytest.mark.parametrize("steps,ds", [(64, 1.0), (24, 7.0), (40, -2.0), (256, 16.0)])
def test_weighted_sides_and_sums(cv, gpu_ctx, N, levels, steps, ds):
    scene = _scene(cv, N, levels, steps, ds)
    log(f"[weighted] N={N} levels={levels} steps={steps} ds={ds}")
    o = run_oracle(scene, want_f64=False)
    g = run_gpu(cv, scene, ctx=gpu_ctx)
    for k, (a, b) in enumerate(zip(g.levels, o.levels)):
        assert_bit_equal(f"level {k}", a, b)
    assert_bit_equal("image", g.image, o.img32)


@pytest.mark.parametrize("offset", [-2.0, 1.5, 9.0])
def test_weighted_lod_offset(cv, gpu_ctx, offset):
    scene = _scene(cv, 32, 6, 48, 16.0, offset=offset)
    log(f"[weighted] lod offset {offset}")
    assert_bit_equal("image", run_gpu(cv, scene, ctx=gpu_ctx).image, run_oracle(scene, want_f64=False).img32)


def test_weighted_frames_reuse_slots(cv, gpu_ctx):
    """Frames of moving clouds in one volume equal the same frames in volumes
    of their own: slots a frame leaves empty hold nothing of an earlier one."""
    import torch
    scene = _scene(cv, 48, 6, 64, 16.0)
    log("[weighted] five frames in one volume")
    vol, sun, cam, vox, tr = cv.scene_objects(scene, context=gpu_ctx)
    try:
        for f in range(5):
            xyz = (scene.xyz + np.float32(0.35 * (f - 2))).astype(np.float32)
            img = torch.zeros((scene.H, scene.W, 4), dtype=torch.float32, device="cuda")
            vol.set_billboards(xyz, scene.scales)
            vox.voxelize(vol, sun)
            tr.coneTrace(vol, sun, cam, img, scene.W, scene.H)
            torch.cuda.synchronize()
            fresh = run_gpu(cv, replace(scene, xyz=xyz), ctx=gpu_ctx)
            assert_bit_equal(f"frame {f}", img.cpu().numpy(), fresh.image)
    finally:
        vol.close()


@pytest.mark.parametrize("kw", [dict(octaves=1), dict(octaves=16, pers_step=0.9, freq_step=2.0),
                                dict(octaves=6, pers_step=1e6), dict(octaves=4, adjust_size=1e-9),
                                dict(octaves=3, offsets=(2e9, -3e9, 0.5)), dict(octaves=5, freq_step=-300.0),
                                dict(min_steps=1, max_steps=2), dict(color_scale=-0.5, min_color=-0.1)])
def test_noise_march_params(cv, gpu_ctx, kw):
    scene = replace(_scene(cv, 32, 6, 16, 1.0), noise_march=cv.scenes.NoiseMarch(seed=3, **kw))
    log(f"[noise march] {kw}")
    assert_bit_equal("image", run_gpu(cv, scene, ctx=gpu_ctx).image, run_oracle(scene, want_f64=False).img32)
