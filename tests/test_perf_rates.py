"""The rates that imexlb.perf reports count the bytes of a pass once, however
many steps the pass makes."""
import pytest

from imexlb import perf


def test_bytes_per_update():
    assert perf.bytes_per_update(27, 8, 1) == 432
    assert perf.bytes_per_update(9, 8, 2) == 72
    assert perf.bytes_per_update(9, 2, 5) == 7.2


@pytest.mark.gpu
def test_no_rate_above_the_memory_s_peak():
    """8192x2048 FP64 makes two steps per pass; counted by the step, its rate
    was 10 TB/s."""
    print("[perf] 8192x2048 f64", flush=True)
    r = perf.measure("cyl8192x2048", "f64", seconds=0.1, timed_steps=41)
    assert r["form"] == "f64" and r["steps_per_pass"] == 2 and r["algorithmic_bytes_per_update"] == 72
    assert 0.3 < r["frac_of_peak"] < 1.0, r
