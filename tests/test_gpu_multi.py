"""Several steps per launch (small 2D lattices) against one step per launch
and against the oracle: the same bits.  IMEXLB_MULTI=0 keeps single steps."""
import numpy as np
import pytest

import imexlb as I
from cases import assert_state_equal, get_deck, oracle_setup

pytestmark = pytest.mark.gpu
PRECS = {"f64": I.F64, "f32": I.F32, "f16": I.F16_F32, "bf16": I.BF16_F32, "bf16sr": I.BF16SR_F32}


def _deck(d):
    if isinstance(d, str):
        return get_deck(d)
    nx, ny = d
    dia = max(2.0, 0.2 * ny)
    return I.Deck(2, (nx, ny, 0), dia / nx, 0.3, 50.0, 1.0 / (3.0 * 0.05 * dia / 50.0 + 0.5), 1.0, 1.0, 1.0, 0.01)


def _pair(monkeypatch, deck, prec, shape=None):
    rv = np.random.default_rng(3).random(100)
    out = []
    for multi in ("1", "0"):
        monkeypatch.setenv("IMEXLB_MULTI", multi)
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


# one window and several, axes around the 32 cells of a window and the 50 of
# two, the thinnest channel, the body near a wall, cut by the inlet, turned
DECKS = [("tiny2d", None), ("ragged2d", None), ("inletbody2d", None), ("channel3", None), ("input.in", (1.7, 30.0)),
         ((2, 2), None), ((30, 31), None), ((31, 32), None), ((32, 49), None), ((49, 50), None), ((50, 67), None),
         ((68, 24), None), ((255, 64), None)]


@pytest.mark.parametrize("deck,shape", DECKS)
@pytest.mark.parametrize("prec", ["f64", "f16"])
def test_multi_steps_equal_single_steps(monkeypatch, deck, shape, prec):
    print(f"[multi] {deck} {shape} {prec}", flush=True)
    a, b = _pair(monkeypatch, _deck(deck), PRECS[prec], shape)
    for n in (1, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 36, 250):
        a.advance(n)
        b.advance(n)
        _same(a, b)
    a.close()
    b.close()


@pytest.mark.parametrize("prec", list(PRECS))
def test_multi_steps_in_every_storage_form(monkeypatch, prec):
    a, b = _pair(monkeypatch, _deck((300, 90)), PRECS[prec])
    a.advance(203)
    b.advance(203)
    _same(a, b)
    for lat in (a, b):  # new parameters, phase by phase, then together
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
    for lat in (a, b):  # timed launches
        lat.profile(True)
        lat.advance(50)
        lat.synchronize()
        assert lat.profile_read()[0][0] == 50
        lat.profile(False)
    _same(a, b)
    a.close()
    b.close()


# lattices that take windows of two and four cells per thread
@pytest.mark.parametrize("n,prec", [((900, 225), "f32"), ((900, 225), "f16"), ((2999, 301), "f32"),
                                    ((3601, 1003), "f16"), ((3601, 1003), "bf16")])
def test_large_windows_equal_other_forms(monkeypatch, n, prec):
    print(f"[multi] {n} {prec}", flush=True)
    a, b = _pair(monkeypatch, _deck(n), PRECS[prec])
    for lat in (a, b):
        lat.advance(22)
    _same(a, b)
    a.close()
    b.close()


@pytest.mark.parametrize("name", ["tiny2d", "inletbody2d", "ragged2d", "channel3", "input.in"])
def test_multi_steps_match_oracle(name):
    rv = np.random.default_rng(4).random(100)
    deck = get_deck(name)
    lat, _ = I.setup(deck, rv, device=0)
    o, _ = oracle_setup(deck, rv)
    lat.advance(41)
    o.run(0, 40, 0)
    assert_state_equal(lat, o)
    lat.close()
    o.close()


@pytest.mark.parametrize("prec", ["f64", "f32", "f16"])
def test_ensemble_multi_steps_equal_single_steps(monkeypatch, prec):
    """Uneven cases, one within a window and one with a turned ellipse."""
    from imexlb.ensemble import Batch, cylinder_cases
    out = []
    for multi in ("1", "0"):
        monkeypatch.setenv("IMEXLB_MULTI", multi)
        b = Batch([_deck(n) for n in ((28, 24), (61, 20), (150, 60), (90, 33))] + cylinder_cases(3, seed=2),
                  precision=PRECS[prec])
        b.init(np.linspace(0.0, 1.0, 100))
        res = []
        for n in (1, 4, 5, 12, 131):
            b.advance(n)
            res.append([b.forces(), b.monitor()[0]] + [v for i in range(b.ncase) for v in b.download_fields(i)])
        b.init(np.linspace(1.0, 0.0, 100))
        b.advance(60)
        res.append([v for i in range(b.ncase) for v in b.download_fields(i)])
        out.append(res)
        del b
    for r, s in zip(*out):
        for x, y in zip(r, s):
            assert np.array_equal(x, y)
