"""The device memory of the forms that make several steps at a time: a plan
that gets none leaves single steps behind, not an error, and what a plan keeps
is part of the device bytes that a lattice or an ensemble reports."""
import ctypes as C

import numpy as np
import pytest

import imexlb as I
import test_gpu_multi as M
from imexlb.ensemble import Batch

pytestmark = pytest.mark.gpu
# a 2D lattice makes 10 allocations at creation and 11 in SetGeometry before
# those of a plan (4 for several steps per launch, 5 for two per pass)
FIRST, MULTI, DOUBLE = 22, 4, 5


def _lattice(deck):
    d = I.derive(deck)
    lat = I.Lattice(2, *deck.n[:2], device=0)
    lat.set_params(deck.ome, deck.rho0, d.uu)
    lat.set_geometry(d.pos, d.radius)
    lat.init_up(np.linspace(0.0, 1.0, 100))
    lat.init_pdf()
    lat.advance(33)
    out = lat.step_form()["steps_per_pass"], lat.info(), lat.download_pdf(I.PDF_F)
    lat.set_geometry(d.pos, d.radius)  # (the hook fails one allocation only)
    return *out, lat.step_form()["steps_per_pass"], lat.close()


@pytest.mark.parametrize("form,count", [("multi", MULTI), ("double", DOUBLE)])
def test_plan_without_memory_leaves_single_steps(monkeypatch, form, count):
    deck = M._deck((300, 90))
    if form == "double":
        monkeypatch.setenv("IMEXLB_SMALL_CELLS", "0")
        monkeypatch.setenv("IMEXLB_MULTI", "0")
    steps, full, f, *_ = _lattice(deck)
    assert (steps >= 3) if form == "multi" else (steps == 2)
    left = set()
    for at in range(FIRST, FIRST + count):
        print(f"[plan] {form}: allocation {at} fails", flush=True)
        monkeypatch.setenv("IMEXLB_FAIL_ALLOC", str(at))
        n, info, g, again, _ = _lattice(deck)
        assert n == 1 and again == steps
        assert (f == g).all()
        left.add(info["device_bytes"])
    assert len(left) == 1
    kept = full["device_bytes"] - left.pop()
    assert kept >= (9 * full["plane_bytes"] if form == "double" else 4)
    monkeypatch.setenv("IMEXLB_FAIL_ALLOC", str(FIRST + count))  # the first one of the next SetGeometry
    with pytest.raises(I.ImexlbError) as err:
        _lattice(deck)
    assert err.value.code == I.E_OOM


def _batch(decks):
    b = Batch(decks)
    info = (C.c_int64 * 4)()
    assert I.lib().imexlb_batch_info(b._h, info) == 0
    b.init(np.linspace(0.0, 1.0, 100))
    b.advance(33)
    out = b.step_form()["steps_per_pass"], info[3], [b.download_fields(i) for i in range(len(decks))]
    b.close()
    return out


def test_ensemble_plan_without_memory_leaves_single_steps(monkeypatch):
    decks = [M._deck(n) for n in ((28, 24), (61, 20), (150, 60))]
    steps, full, f = _batch(decks)
    assert steps >= 3
    left = set()
    for at in range(22, 29):
        print(f"[plan] ensemble: allocation {at} fails", flush=True)
        monkeypatch.setenv("IMEXLB_FAIL_ALLOC", str(at))
        n, bytes_, g = _batch(decks)
        assert n == 1
        for (p, u), (q, v) in zip(f, g):
            assert (p == q).all() and (u == v).all()
        left.add(bytes_)
    assert len(left) == 1 and full > left.pop()
    for at in (1, 21):
        monkeypatch.setenv("IMEXLB_FAIL_ALLOC", str(at))
        with pytest.raises(I.ImexlbError) as err:
            Batch(decks)
        assert err.value.code == I.E_OOM
    monkeypatch.setenv("IMEXLB_FAIL_ALLOC", "29")
    assert _batch(decks)[0] == steps
