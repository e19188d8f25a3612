"""Short runs of steps on the lattices that do not take three steps per launch,
nor short runs in several: against single steps, bit for bit."""
import numpy as np
import pytest

import imexlb as I
import test_gpu_multi as M

pytestmark = pytest.mark.gpu


# above the size from which a launch makes five steps or none; mostly windows
# with tables (short runs in single steps); small: three steps and two singles
@pytest.mark.parametrize("n,prec", [((1500, 900), "f16"), ((60, 24000), "f64"), ((60, 75000), "f16"), ((400, 100), "f32")])
def test_short_runs_equal_single_steps(monkeypatch, n, prec):
    print(f"[short] {n} {prec}", flush=True)
    lats = []
    for multi in ("1", "0"):
        monkeypatch.setenv("IMEXLB_MULTI", multi)
        monkeypatch.setenv("IMEXLB_DOUBLE", "0")
        lat = I.Lattice(2, *n, device=0, precision=M.PRECS[prec])
        lat.set_params(1.5, 1.0, 0.02)
        lat.set_geometry(0.4 * n[0], 0.1 * min(n))
        lat.init_up(np.linspace(0.0, 1.0, 100))
        lat.init_pdf()
        lats.append(lat)
    a, b = lats
    assert a.step_form()["steps_per_pass"] >= 3 and b.step_form()["steps_per_pass"] == 1
    for k in (2, 3, 4, 5, 6, 7, 8, 9, 11, 16, 23):
        for lat in lats:
            lat.advance(k)
        assert np.array_equal(a.forces(), b.forces()), k
    for x, y in zip(a.download_fields(), b.download_fields()):
        assert np.array_equal(x, y, equal_nan=True)
    assert np.array_equal(a.download_pdf(I.PDF_FB), b.download_pdf(I.PDF_FB), equal_nan=True)
    a.close()
    b.close()
