"""The footprint slots of R8 volumes: made by the first cone trace and not
before, given back with the volume; and the same cones without them
(CR_CONTEXT_DIRECT_ADDRESSING), against the oracle's FP32 pass bit for bit."""
import time
from dataclasses import replace

import numpy as np
import pytest

from gpu_common import assert_bit_equal, log, run_gpu, run_oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def direct_ctx(cv):
    ctx = cv.Context(0, flags=cv._abi.CR_CONTEXT_DIRECT_ADDRESSING)
    yield ctx
    ctx.close()


def _scene(cv, N, levels, steps, ds, **kw):
    base = cv.scenes.reference_mode(cv.scenes.small32(N))
    cone = replace(base.cone, steps=steps, down_scaling=ds, cone_angle=0.6, quantize_rgba8=0, **kw)
    return replace(base, N=N, levels=levels, W=72, H=40, light_w=128, light_h=128, cone=cone)


@pytest.mark.parametrize("direct", [False, True])
def test_memory(cv, gpu_ctx, direct_ctx, direct):
    import torch

    log(f"[slots] memory, direct addressing {direct}")
    N = 256
    slots = 8 * sum((N >> k) ** 3 for k in range(9))
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    scene = _scene(cv, N, 9, 16, 1.0)
    img = torch.zeros((scene.H, scene.W, 4), dtype=torch.float32, device="cuda")
    free0 = torch.cuda.mem_get_info()[0]
    vol, sun, cam, vox, tr = cv.scene_objects(scene, context=direct_ctx if direct else gpu_ctx)
    try:
        for _ in range(2):
            vox.voxelize(vol, sun)
        torch.cuda.synchronize()
        made = free0 - torch.cuda.mem_get_info()[0]
        assert made < slots, "voxelizing alone takes the slots' memory"
        tr.coneTrace(vol, sun, cam, img, scene.W, scene.H)
        torch.cuda.synchronize()
        traced = free0 - torch.cuda.mem_get_info()[0]
        assert (traced - made < slots) if direct else (2 * slots <= traced - made < 3 * slots)
    finally:
        vol.close()
    # the driver may report freed memory a little later
    for _ in range(40):
        held = free0 - torch.cuda.mem_get_info()[0]
        if held < slots:
            break
        time.sleep(0.05)
    assert held < slots


@pytest.mark.parametrize("N,levels", [(1, 1), (3, 1), (5, 3), (17, 5), (48, 6), (64, 7)])
@pytest.mark.parametrize("steps,ds", [(64, 1.0), (40, -2.0), (256, 16.0)])
@pytest.mark.parametrize("composite", [0, 1])
def test_without_slots(cv, direct_ctx, N, levels, steps, ds, composite):
    scene = _scene(cv, N, levels, steps, ds, composite=composite)
    log(f"[slots] texels: N={N} levels={levels} steps={steps} ds={ds} composite={composite}")
    assert_bit_equal("image", run_gpu(cv, scene, ctx=direct_ctx).image, run_oracle(scene, want_f64=False).img32)


@pytest.mark.parametrize("kw", [dict(octaves=3), dict(octaves=6, pers_step=1e6), dict(color_scale=-0.5, min_color=-0.1)])
def test_noise_march_without_slots(cv, direct_ctx, kw):
    scene = replace(_scene(cv, 32, 6, 16, 1.0), noise_march=cv.scenes.NoiseMarch(seed=3, **kw))
    log(f"[slots] texels, noise march {kw}")
    assert_bit_equal("image", run_gpu(cv, scene, ctx=direct_ctx).image, run_oracle(scene, want_f64=False).img32)


@pytest.mark.parametrize("before", [1, 2, 3])
def test_first_trace_between_frames(cv, gpu_ctx, before):
    """Slots made while frames are queued: voxelizations before the first trace,
    frames of moving clouds after it, nothing waited for in between."""
    import torch

    log(f"[slots] {before} voxelizations before the first trace")
    scene = _scene(cv, 48, 6, 64, 16.0)
    moved = [(scene.xyz + np.float32(0.3 * (f - 2))).astype(np.float32) for f in range(5)]
    want = [run_oracle(replace(scene, xyz=m), want_f64=False).img32 for m in moved]
    vol, sun, cam, vox, tr = cv.scene_objects(scene, context=gpu_ctx)
    try:
        imgs = [torch.zeros((scene.H, scene.W, 4), dtype=torch.float32, device="cuda") for _ in moved]
        for _ in range(before):
            vox.voxelize(vol, sun)
        for m, img in zip(moved, imgs):
            vol.set_billboards(m, scene.scales)
            vox.voxelize(vol, sun)
            tr.coneTrace(vol, sun, cam, img, scene.W, scene.H)
        torch.cuda.synchronize()
        for f, img in enumerate(imgs):
            assert_bit_equal(f"frame {f}", img.cpu().numpy(), want[f])
    finally:
        vol.close()


@pytest.mark.parametrize("light", [128, 1024])
def test_first_trace_on_another_stream(cv, gpu_ctx, light):
    """The next frame's voxelization on its own stream, beside a first trace that
    is still queued on another (side streams in a chain and apart)."""
    import torch

    log(f"[slots] first trace on another stream, light {light}")
    scene = replace(_scene(cv, 48, 6, 64, 16.0), light_w=light, light_h=light)
    moved = [scene.xyz, (scene.xyz + np.float32(0.4)).astype(np.float32)]
    want = [run_oracle(replace(scene, xyz=m), want_f64=False).img32 for m in moved]
    for _ in range(2):
        vol, sun, cam, vox, tr = cv.scene_objects(scene, context=gpu_ctx)
        try:
            a, b = torch.cuda.Stream(), torch.cuda.Stream()
            imgs = [torch.zeros((scene.H, scene.W, 4), dtype=torch.float32, device="cuda") for _ in moved]
            torch.cuda.synchronize()
            for q in range(2):  # both level sets exist
                vox.voxelize(vol, sun, stream=a)
            b.wait_stream(a)
            with torch.cuda.stream(b):
                torch.cuda._sleep(20_000_000)
            tr.coneTrace(vol, sun, cam, imgs[0], scene.W, scene.H, stream=b)
            vol.set_billboards(moved[1], scene.scales)
            vox.voxelize(vol, sun, stream=a)
            tr.coneTrace(vol, sun, cam, imgs[1], scene.W, scene.H, stream=a)
            torch.cuda.synchronize()
            for f, img in enumerate(imgs):
                assert_bit_equal(f"frame {f}", img.cpu().numpy(), want[f])
        finally:
            vol.close()
