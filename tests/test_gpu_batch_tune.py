"""The ensemble's shape tuner times the kernel whose shape it chooses."""
import numpy as np
import pytest

import test_gpu_multi as M

pytestmark = pytest.mark.gpu


def test_tuner_times_single_steps():
    """Launches of several steps take 1.3 us a step here, single steps 3.5 and
    more whatever their shape."""
    import time

    from imexlb.ensemble import Batch
    b = Batch([M._deck(n) for n in ((28, 24), (61, 20), (90, 33))])
    form = b.step_form()
    assert form["steps_per_pass"] >= 3
    b.init(np.linspace(0.0, 1.0, 100))
    best = b.tune(40)
    assert b.step_form() == form  # as it was
    per = 1e9
    for _ in range(5):
        b.synchronize()
        t = time.perf_counter()
        b.advance(4001)
        b.synchronize()
        per = min(per, (time.perf_counter() - t) / 4001 * 1e3)
    print(f"[tune] {best}, several per launch {per * 1e3:.2f} us", flush=True)
    assert best["ms_per_step"] > 1.6 * per
    b.close()
