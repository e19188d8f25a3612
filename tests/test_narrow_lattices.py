"""Narrow and tall 2D lattices: rows are padded to whole 64-cell tiles only
where two steps per pass use them, and the step's form goes by the cells of
the lattice, not of its padding."""
import numpy as np
import pytest

import imexlb as I

U = 0.05


def test_a_tall_lattice_is_not_refused_for_its_padding():
    """20 x 60,000,000 FP16 nodes have fewer than 2^31 cells (1.4e9); with
    rows of 64 cells they would have more."""
    import ctypes as C
    n = C.c_int()
    I.lib().imexlb_device_count(C.byref(n))
    if n.value:
        pytest.skip("would allocate the lattice")
    with pytest.raises(I.ImexlbError) as err:
        I.Lattice(2, 20, 60_000_000, 0, device=0, precision=I.F16_F32)
    assert "too large" not in str(err.value), err.value


# size, precision, steps per pass (0: several per launch), row cells
FORMS = [((20, 100_000), I.F64, 0, 23), ((20, 130_000), I.F64, 1, 23), ((700, 13_000), I.F16_F32, 1, 703),
         ((100, 40_000), I.F64, 1, 103),
         ((180, 20_000), I.F64, 2, 192), ((300, 9_000), I.F64, 2, 320), ((2000, 1500), I.F64, 2, 2048),
         ((20, 200_000), I.F32, 0, 23), ((400, 12_000), I.F32, 0, 403), ((2800, 1500), I.F32, 0, 2816),
         ((130, 46_000), I.F16_F32, 0, 133), ((100, 100_000), I.F16_F32, 1, 103), ((1000, 9_000), I.BF16_F32, 2, 1024),
         ((2000, 5_000), I.F16_F32, 2, 2048), ((520, 12_000), I.BF16SR_F32, 1, 523), ((10, 200_000), I.F64, 0, 13)]


@pytest.mark.gpu
@pytest.mark.parametrize("n,prec,steps,row", FORMS)
def test_form_and_rows_of_narrow_lattices(monkeypatch, n, prec, steps, row):
    print(f"[narrow] {n} {prec}", flush=True)
    fields = []
    for off in (False, True):
        if off:
            monkeypatch.setenv("IMEXLB_DOUBLE", "0")
            monkeypatch.setenv("IMEXLB_MULTI", "0")
        lat = I.Lattice(2, *n, 0, device=0, precision=prec)
        lat.set_params(1.7, 1.0, U)
        lat.set_geometry(0.5 * n[0], 0.12 * n[0])
        if not off:
            f = lat.step_form()
            assert f["row_cells"] == row, f
            assert (f["steps_per_pass"] >= 3) if steps == 0 else (f["steps_per_pass"] == steps), f
        lat.init_up(np.linspace(0.0, 1.0, 100))
        lat.init_pdf()
        lat.advance(21)
        fields.append(lat.download_fields())
        lat.close()
    for a, b in zip(*fields):  # (the inlet profile of the tallest overflows the integer ny*ny: NaN in both)
        assert np.array_equal(a, b, equal_nan=True)
