"""Uploads of billboards right behind a queued batch run: the run still reads the
billboards it was called with, on the default stream and on a stream of the
caller's own, also where an upload of no billboards comes in between."""
from dataclasses import replace

import numpy as np
import pytest

from gpu_common import assert_bit_equal, log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("own_stream", [False, True])
@pytest.mark.parametrize("empty_first", [False, True])
def test_upload_behind_a_batch(cv, gpu_ctx, own_stream, empty_first):
    import torch

    log(f"[upload order] own stream {own_stream}, empty upload first {empty_first}")
    scenes = [replace(s, W=128, H=128, light_w=128, light_h=128) for s in cv.scenes.batched64(5, count=3)]
    rng = np.random.default_rng(11)
    entries = []
    for sc in scenes:
        vol, sun, cam, vox, tr = cv.scene_objects(sc, 0, context=gpu_ctx)
        img = torch.full((sc.H, sc.W, 4), -1.0, dtype=torch.float32, device="cuda")
        entries.append((vol, sun, cam, tr, img, vox))
    batch = cv.Batch(entries, context=gpu_ctx)
    try:
        batch.run()
        torch.cuda.synchronize()
        want = [e[4].cpu().numpy() for e in entries]
        stream = torch.cuda.Stream() if own_stream else torch.cuda.current_stream()
        for _ in range(2):
            for e in entries:
                e[4].fill_(-1.0)
            batch.run()  # captures again after the last round's uploads
            torch.cuda.synchronize()
            with torch.cuda.stream(stream):
                torch.cuda._sleep(20_000_000)  # the run is still queued when the uploads come
                batch.run(stream=stream)
            for e, sc in zip(entries, scenes):
                if empty_first:
                    e[0].set_billboards(np.zeros((0, 3), np.float32), np.zeros(0, np.float32))
                e[0].set_billboards(rng.uniform(-0.9, 0.9, size=(sc.S, 3)), np.full(sc.S, 0.2, np.float32))
            torch.cuda.synchronize()
            for q, e in enumerate(entries):
                assert_bit_equal(f"scene {q}", e[4].cpu().numpy(), want[q])
            for e, sc in zip(entries, scenes):
                e[0].set_billboards(sc.xyz, sc.scales)
    finally:
        batch.close()
        for e in entries:
            e[0].close()


def test_mark_outlives_the_batch(cv, gpu_ctx):
    """A volume whose batch is gone takes uploads and frames as before."""
    import torch

    log("[upload order] upload after the batch was destroyed")
    sc = replace(cv.scenes.batched64(5, count=1)[0], W=128, H=128, light_w=128, light_h=128)
    vol, sun, cam, vox, tr = cv.scene_objects(sc, 0, context=gpu_ctx)
    img = torch.zeros((sc.H, sc.W, 4), dtype=torch.float32, device="cuda")
    try:
        batch = cv.Batch([(vol, sun, cam, tr, img, vox)], context=gpu_ctx)
        batch.run()
        torch.cuda.synchronize()
        want = img.cpu().numpy()
        batch.close()
        vol.set_billboards(sc.xyz, sc.scales)
        img.fill_(-1.0)
        vox.voxelize(vol, sun)
        tr.coneTrace(vol, sun, cam, img, sc.W, sc.H)
        torch.cuda.synchronize()
        assert_bit_equal("image", img.cpu().numpy(), want)
    finally:
        vol.close()
