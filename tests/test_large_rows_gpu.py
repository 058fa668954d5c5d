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


def test_forward(cv, gpu_ctx):
    import torch

    n, edge = (1 << 31) - 100, 3000
    log(f"[large rows] forward of {n} rows")
    _need(n * (17 + 5) * 4)
    g = torch.Generator(device="cuda")
    g.manual_seed(2)
    mlp = cv.FarFieldMLP(context=gpu_ctx, params=cv.FarFieldMLP.init_params(3))
    x = torch.zeros((n, 17), device="cuda")
    # random rows at both ends and around the middle, zeros between
    at = [0, (n >> 1) - edge, (1 << 30) - edge // 2, n - edge]
    for a in at:
        x[a:a + edge] = torch.rand((edge, 17), generator=g, device="cuda")
    y = mlp.forward(x)
    try:
        for a in at:
            want = mlp.forward(x[a:a + edge].clone())
            assert torch.equal(y[a:a + edge].view(torch.int32), want.view(torch.int32)), f"rows from {a}"
        zero = mlp.forward(torch.zeros((1, 17), device="cuda"))
        assert torch.equal(y[n // 3:n // 3 + 5], zero.expand(5, -1))
    finally:
        del x, y
        torch.cuda.empty_cache()
