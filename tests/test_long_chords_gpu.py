"""Pass 1 with billboards of thousands of voxels' radius in elongated volumes,
which reach chord samples beyond 2^15: chords just below and above the lengths
up to which they are cut into depth slices, with an exact (power-of-two) and an
accumulated step.  The occupancy is the oracle's, voxel for voxel."""
from dataclasses import replace

import numpy as np
import pytest

import oracle_lib as O
from gpu_common import log, run_gpu

pytestmark = pytest.mark.gpu


# side, radius in steps
@pytest.mark.parametrize("N,steps", [(96, 1990.0), (96, 2050.0), (96, 20000.0), (96, 32700.0), (96, 33000.0),
                                     (150, 32760.0), (64, 20000.0), (64, 32700.0), (64, 33000.0)])
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_far_half_of_the_chord(cv, gpu_ctx, N, steps, sign):
    log(f"[long chords] N={N} radius {steps} steps, sun {sign}")
    half = np.array([1.0, 1.0, 128.0])
    step = 2.0 / N
    # centres towards either end of the volume, on its axis: with the sun along
    # it the volume lies in the near or the far half of the chords
    xyz = np.array([[0.1, -0.2, 90.0], [-0.3, 0.1, -100.0], [0.0, 0.0, 0.0]], np.float32)
    r = np.array([steps, steps * 0.999, 3.0], np.float32) * np.float32(step)
    base = cv.scenes.small32(1)
    for order in ([0, 2], [1, 2]):
        sc = replace(base, N=N, levels=cv.scenes.full_levels(N), xyz=xyz[order], scales=r[order],
                     sun_dir=np.array([0.0, 0.0, sign]), W=16, H=16, light_w=1025, light_h=3, bounds_lo=tuple(-half),
                     bounds_hi=tuple(half), cone=replace(base.cone, steps=4))
        want = O.voxelize(sc).state()
        assert want.any()
        g = run_gpu(cv, sc, ctx=gpu_ctx, read_levels=False)
        assert np.array_equal(g.state, want)
