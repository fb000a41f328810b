"""The autotuner's choice for a plan of few slices is not taken over by one of
many: timing 7 to 14 shapes rebuilds the plan's tables as often, taking over a
cached choice rebuilds them once, so the time of the call tells which it was."""
import time

import numpy as np
import pytest

from aretomo3_amd import Plan
from aretomo3_amd import _lib as L

pytestmark = pytest.mark.gpu


def timed(plan):
    t0 = time.perf_counter()
    choice = plan.autotune()
    return time.perf_counter() - t0, choice


@pytest.mark.parametrize("px,storage", [(1024, L.STORAGE_F32), (640, L.STORAGE_BF16)])
def test_many_slices_are_timed_for_themselves(gpu_available, px, storage):
    tilts = np.linspace(-60.0, 60.0, 31).astype(np.float32)
    kw = dict(sart_iters=1, sart_subsets=3, positivity=False, storage=storage)
    print(f"case autotune {px}, storage {storage}", flush=True)
    few = Plan(px, 2, tilts, 75, L.METHOD_SART, **kw)
    many = Plan(px, 500, tilts, 75, L.METHOD_SART, **kw)
    few.autotune()
    first, choice = timed(many)
    cached = []
    for _ in range(3):
        t, again = timed(many)
        assert again == choice
        cached.append(t)
    print(f"first call {1e3 * first:.1f} ms, cached {1e3 * min(cached):.1f} ms")
    assert first > 3 * min(cached)
