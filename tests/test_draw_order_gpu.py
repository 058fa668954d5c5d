"""Draw orders against the oracle's literal selection sort at the sizes where
the sort changes form (one workgroup up to 1024 billboards, counting in chunks
of 512 up to 16384, beyond in memory) and at every amount of equal distances:
none, a few short runs (resolved on demand), many or long ones (every step
replayed)."""
from dataclasses import replace

import numpy as np
import pytest

import oracle_lib as O
from gpu_common import log

pytestmark = pytest.mark.gpu


def _positions(S, ties, rng):
    """Offsets whose distances from the origin repeat as asked."""
    p = rng.uniform(-1.0, 1.0, size=(S, 3)).astype(np.float32)
    n = min(S, {"none": 0, "few": max(2, S // 200), "many": S // 2, "all": S}[ties])
    if ties == "all":
        p[:] = (0.5, 0.25, -0.25)
    else:
        at = rng.choice(S, size=n - n % 2, replace=False)
        p[at[0::2]] = p[at[1::2]]          # equal pairs
        if ties == "many" and S >= 64:
            p[rng.choice(S, size=40, replace=False)] = p[0]  # and one run of 40
        if ties == "few" and S >= 1024:
            p[rng.choice(S, size=9, replace=False)] = p[1]   # and one of 9 or 10
            near = np.argsort(np.linalg.norm(p, axis=1))[:4]  # and a pair among the last drawn from the origin
            p[near[1]] = p[near[2]]
    return p


@pytest.mark.parametrize("ties", ["none", "few", "many", "all"])
@pytest.mark.parametrize("S", [1, 2, 63, 513, 1024, 1025, 2047, 4096, 5000, 15361, 16384, 16385])
def test_order(cv, gpu_ctx, S, ties):
    if ties == "all" and S > 2100:
        pytest.skip("a run of every billboard takes the oracle and the replay O(S^2)")
    if ties == "many" and S > 16384:
        pytest.skip("the replay in memory walks thousands of runs on one thread")
    rng = np.random.default_rng(S)
    p = _positions(S, ties, rng)
    scene = replace(cv.scenes.small32(0), xyz=p, scales=np.full(S, 0.05, np.float32))
    eye = (0.0, 0.0, 0.0) if S % 2 else tuple(float(x) for x in p[S // 2])  # also a distance of exactly 0
    log(f"[order] S={S} ties={ties}")
    vol, _, _, _, _ = cv.scene_objects(scene, context=gpu_ctx)
    try:
        got = vol.sortBoards(eye)
    finally:
        vol.close()
    assert np.array_equal(got, O.sort_boards(scene, eye))
