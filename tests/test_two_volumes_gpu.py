"""Two volumes of one context drawn in turn, one small enough for its passes to
follow one another on one side stream, the other on three: every image is the
one of its own volume's billboards, with uploads in between and without."""
from dataclasses import replace

import numpy as np
import pytest

from gpu_common import assert_bit_equal, log, run_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("uploads", [False, True])
def test_in_turn(cv, gpu_ctx, uploads):
    import torch

    log(f"[two volumes] uploads {uploads}")
    base = cv.scenes.small32(21)
    scenes = [base, replace(base, N=64, levels=cv.scenes.full_levels(64), light_w=900, light_h=700, fmt=2)]
    shift = [np.float32(0.0), np.float32(0.2), np.float32(-0.2)] if uploads else [np.float32(0.0)] * 3
    want = [[run_oracle(replace(s, xyz=s.xyz + d), want_f64=False).img32 for d in shift] for s in scenes]
    objs = [cv.scene_objects(s, 0, context=gpu_ctx) for s in scenes]
    try:
        imgs = [[torch.zeros((s.H, s.W, 4), dtype=torch.float32, device="cuda") for _ in shift] for s in scenes]
        for _ in range(2):
            for f, d in enumerate(shift):
                for (vol, sun, cam, vox, tr), s, im in zip(objs, scenes, imgs):
                    if uploads:
                        vol.set_billboards(s.xyz + d, s.scales)
                    vox.voxelize(vol, sun)
                    tr.coneTrace(vol, sun, cam, im[f], s.W, s.H)
            torch.cuda.synchronize()
            for q in range(2):
                for f in range(len(shift)):
                    assert_bit_equal(f"volume {q} frame {f}", imgs[q][f].cpu().numpy(), want[q][f])
    finally:
        for o in objs:
            o[0].close()
