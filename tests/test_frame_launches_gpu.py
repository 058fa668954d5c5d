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


@pytest.mark.parametrize("own_stream", [False, True])
def test_uploads_between_frames(cv, gpu_ctx, own_stream):
    """New billboards for every frame, nothing waited for in between: each
    image is the one of its own billboards."""
    import torch

    log(f"[launches] uploads between frames, own stream {own_stream}")
    base = cv.scenes.small32(3)
    sets = []
    for q in range(5):
        rng = np.random.default_rng(q)
        S = (300, 7, 1500, 300, 64)[q]
        sets.append((rng.uniform(-0.7, 0.7, size=(S, 3)).astype(np.float32),
                     rng.uniform(0.02, 0.2, size=S).astype(np.float32)))
    want = [run_oracle(replace(base, xyz=x, scales=r), want_f64=False).img32 for x, r in sets]
    vol, sun, cam, vox, tr = cv.scene_objects(base, 0, context=gpu_ctx)
    try:
        for _ in range(2):
            imgs = [torch.zeros((base.H, base.W, 4), dtype=torch.float32, device="cuda") for _ in sets]
            stream = torch.cuda.Stream() if own_stream else torch.cuda.current_stream()
            stream.wait_stream(torch.cuda.current_stream())
            for (x, r), img in zip(sets, imgs):
                vol.billboards.positions, vol.billboards.scales = x, r
                vol.update()
                vox.voxelize(vol, sun, stream=stream)
                tr.coneTrace(vol, sun, cam, img, base.W, base.H, stream=stream)
            torch.cuda.synchronize()
            for q, img in enumerate(imgs):
                assert_bit_equal(f"image {q}", img.cpu().numpy(), want[q])
    finally:
        vol.close()


def test_alternating_light_sizes(cv, gpu_ctx):
    """Frames of one volume that change between one side stream and three (the
    light image's size decides): each image is the one of its own light image."""
    import torch

    log("[launches] one and three side streams in turn")
    base = cv.scenes.small32(9)
    sizes = [256, 1024, 256, 256, 1024, 1024, 256, 1024]
    want = {n: run_oracle(replace(base, light_w=n, light_h=n), want_f64=False).img32 for n in set(sizes)}
    vol, _, cam, vox, tr = cv.scene_objects(base, 0, context=gpu_ctx)
    try:
        suns, imgs = [], []
        for n in sizes:
            _, sun, _, vox_n, _ = cv.scene_objects(replace(base, light_w=n, light_h=n), 0, context=gpu_ctx)
            img = torch.zeros((base.H, base.W, 4), dtype=torch.float32, device="cuda")
            suns.append((sun, vox_n))
            imgs.append(img)
        torch.cuda.synchronize()
        for _ in range(2):
            for (sun, vox_n), img in zip(suns, imgs):
                vox_n.voxelize(vol, sun, stream=torch.cuda.current_stream())
                tr.coneTrace(vol, sun, cam, img, base.W, base.H)
            torch.cuda.synchronize()
            for n, img in zip(sizes, imgs):
                assert_bit_equal(f"light {n}", img.cpu().numpy(), want[n])
    finally:
        vol.close()
