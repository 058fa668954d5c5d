"""Row counts whose threads pass what one launch takes (2^32): the calls take
them, and every row is the one that a small call gives for the same input."""
import numpy as np
import pytest

from gpu_common import log

pytestmark = pytest.mark.gpu


def _need(nbytes):
    import torch
    free = torch.cuda.mem_get_info()[0]
    if free < nbytes * 1.1:
        pytest.skip(f"needs {nbytes >> 30} GiB of device memory, {free >> 30} free")


def test_segments(cv, gpu_ctx):
    import torch

    base, k = 1 << 12, 8
    n = (1 << 28) + 3 * base
    log(f"[large rows] segments of {n} starts")
    _need(n * (3 + 17 + 5 + 1) * 4 + (4 << 30))
    sc = cv.scenes.small32(2)
    vol, sun, _, vox, tr = cv.scene_objects(sc, 0, context=gpu_ctx)
    try:
        vox.voxelize(vol, sun)
        g = torch.Generator(device="cuda")
        g.manual_seed(1)
        p0 = torch.rand((base, 3), generator=g, device="cuda")
        want = tr.segments(vol, sun, p0, k)
        assert want[2].any() and not want[2].all()
        got = tr.segments(vol, sun, p0.repeat(n // base, 1), k)
        for name, a, w in zip(("features", "targets", "valid"), got, want):
            a = a.view(torch.int32).view(n // base, *w.shape)
            w = w.view(torch.int32)
            bad = sum(int((part != w).any()) for part in a.split(4096))
            assert bad == 0, f"{name}: {bad} parts differ"
        del got, a
    finally:
        vol.close()
        torch.cuda.empty_cache()
