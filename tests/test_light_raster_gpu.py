"""Pass 1's queued chord walk on grids whose side is no power of two (the
chord counter accumulates and the index map is one product), at the sizes
where it changes: bitmap words 2048 and 4096, depth slices, chords of more than
256 samples, spheres across the volume's faces, extents other than [-1, 1]^3.
The occupancy is the oracle's, voxel for voxel."""
from dataclasses import replace

import numpy as np
import pytest

from gpu_common import log, run_gpu
import oracle_lib as O

pytestmark = pytest.mark.gpu

# side, world extents, billboards, radius range (in voxels), light image
CASES = {
    "tiny": (10, (2.0, 2.0, 2.0), 20, (0.1, 3.0), 96),
    "odd": (33, (2.0, 2.0, 2.0), 60, (0.3, 6.0), 200),
    "n96": (96, (2.0, 2.0, 2.0), 80, (1.0, 9.0), 256),
    "n96_extents": (96, (4.0, 2.0, 8.0), 40, (1.0, 9.0), 256),
    "n192_sliced": (192, (2.0, 2.0, 2.0), 12, (20.0, 90.0), 128),
    "n260_words": (260, (2.0, 2.0, 2.0), 12, (3.0, 40.0), 320),
    "n300_long": (300, (4.0, 4.0, 4.0), 4, (120.0, 190.0), 64),
}


@pytest.mark.parametrize("case", sorted(CASES))
@pytest.mark.parametrize("sun", [(0.3, 0.8, 0.52), (1.0, 0.0, 0.0)])
def test_occupancy(cv, gpu_ctx, case, sun):
    N, ext, S, (r0, r1), light = CASES[case]
    log(f"[raster] {case} N={N} sun={sun}")
    rng = np.random.default_rng(N + S)
    half = np.array(ext) / 2
    xyz = (rng.uniform(-1.05, 1.05, size=(S, 3)) * half).astype(np.float32)
    r = (rng.uniform(r0, r1, size=S) * min(ext) / N).astype(np.float32)
    r[0] = np.float32(2.0 * min(ext) / N)  # a whole number of steps, up to rounding
    sun = np.asarray(sun) / np.linalg.norm(sun)
    base = cv.scenes.small32(1)
    sc = replace(base, N=N, levels=cv.scenes.full_levels(N), xyz=xyz, scales=r, sun_dir=sun, W=16, H=16,
                 light_w=light, light_h=light - 7, bounds_lo=tuple(-half), bounds_hi=tuple(half),
                 cone=replace(base.cone, steps=4))
    g = run_gpu(cv, sc, ctx=gpu_ctx, read_levels=False)
    want = O.voxelize(sc).state()
    assert want.any()
    assert np.array_equal(g.state, want)
