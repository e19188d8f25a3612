"""Two steps in one pass over memory (large lattices) against one step per
pass: the same bits.  IMEXLB_SMALL_CELLS=0 takes small lattices through the
large ones' path; IMEXLB_DOUBLE=0 keeps single steps."""
import numpy as np
import pytest

import imexlb as I
from cases import assert_state_equal, get_deck, oracle_setup

pytestmark = pytest.mark.gpu
PRECS = {"f64": I.F64, "f32": I.F32, "f16": I.F16_F32, "bf16": I.BF16_F32, "bf16sr": I.BF16SR_F32}


def _pair(monkeypatch, deck, prec, shape=None):
    """The same start twice: double steps and single steps."""
    rv = np.random.default_rng(3).random(100)
    out = []
    for double in ("1", "0"):
        monkeypatch.setenv("IMEXLB_SMALL_CELLS", "0")
        monkeypatch.setenv("IMEXLB_DOUBLE", double)
        d = I.derive(deck)
        lat = I.Lattice(deck.dim, *deck.n, device=0, precision=prec)
        lat.set_params(deck.ome, deck.rho0, d.uu)
        lat.set_geometry(d.pos, d.radius, *(shape or (1.0, 0.0)))
        lat.init_up(rv)
        lat.init_pdf()
        out.append(lat)
    return out


def _same(a, b):
    for which in (I.PDF_F, I.PDF_FB):
        x, y = a.download_pdf(which), b.download_pdf(which)
        assert np.array_equal(x, y), (which, int((x != y).sum()))
    for x, y in zip(a.download_fields(), b.download_fields()):
        assert np.array_equal(x, y)
    assert np.array_equal(a.forces(), b.forces())
    assert a.monitor() == b.monitor()


# one strip and several, one segment and several, widths around a strip's 256
# columns and a tile's 64, the body near a wall, cut by the inlet, turned
DECKS_2D = [("tiny2d", None), ("ragged2d", None), ("inletbody2d", None), ("input.in", None), ("input.in", (1.7, 30.0)),
            ((16, 16), None), ((255, 40), None), ((256, 41), None), ((257, 19), None), ((700, 300), None),
            ((62, 500), None), ((1100, 33), None)]


def _deck(d):
    if isinstance(d, str):
        return get_deck(d)
    nx, ny = d
    dia = 0.2 * ny
    return I.Deck(2, (nx, ny, 0), dia / nx, 0.3, 50.0, 1.0 / (3.0 * 0.05 * dia / 50.0 + 0.5), 1.0, 1.0, 1.0, 0.01)


@pytest.mark.parametrize("deck,shape", DECKS_2D)
@pytest.mark.parametrize("prec", ["f64", "f16"])
def test_double_steps_equal_single_steps_2d(monkeypatch, deck, shape, prec):
    print(f"[double] {deck} {shape} {prec}", flush=True)
    a, b = _pair(monkeypatch, _deck(deck), PRECS[prec], shape)
    for n in (1, 4, 5, 6, 7, 13, 150):  # none, one and many passes, every remainder
        a.advance(n)
        b.advance(n)
        _same(a, b)
    a.close()
    b.close()


@pytest.mark.parametrize("prec", list(PRECS))
def test_double_steps_in_every_storage_form(monkeypatch, prec):
    a, b = _pair(monkeypatch, _deck((300, 90)), PRECS[prec])
    a.advance(203)
    b.advance(203)
    _same(a, b)
    # new parameters after a double step, then phase by phase, then again
    for lat in (a, b):
        lat.set_params(1.2, 1.0, 0.04)
        lat.advance(9)
        for _ in range(37):
            lat.collision()
            lat.boundary_condition()
            lat.propagation()
            lat.post_processing()
    _same(a, b)
    for lat in (a, b):  # a new geometry, a new start
        lat.set_geometry(100.0, 12.0)
        lat.init_up(np.linspace(0.0, 1.0, 100))
        lat.init_pdf()
        lat.advance(50)
    _same(a, b)
    a.close()
    b.close()


def test_double_steps_match_oracle_2d(monkeypatch):
    monkeypatch.setenv("IMEXLB_SMALL_CELLS", "0")
    rv = np.random.default_rng(4).random(100)
    for name in ("tiny2d", "inletbody2d", "ragged2d"):
        deck = get_deck(name)
        lat, _ = I.setup(deck, rv, device=0)
        o, _ = oracle_setup(deck, rv)
        lat.advance(41)
        o.run(0, 40, 0)
        assert_state_equal(lat, o)
        lat.close()
        o.close()


def test_double_steps_under_timing(monkeypatch):
    """Timed launches: the same state, every step counted."""
    a, b = _pair(monkeypatch, _deck((300, 90)), I.F64)
    a.profile(True)
    a.advance(50)
    a.synchronize()
    n, ms = a.profile_read()
    a.profile(False)
    b.advance(50)
    assert n[0] == 50 and ms[0] > 0.0
    _same(a, b)
    a.close()
    b.close()
