"""Which form of the time step a lattice or an ensemble takes: that the
comparisons of several steps per launch and of two steps per pass with single
steps compare what they say, and the tests of the single-step forms with the
other two switched off (IMEXLB_MULTI=0, IMEXLB_DOUBLE=0)."""
import pytest

import imexlb as I
import test_gpu_batch as B
import test_gpu_configs as C
import test_gpu_double as D
import test_gpu_multi as M
import test_gpu_parity as P

pytestmark = pytest.mark.gpu

# several steps per launch do not suit a body cut by the inlet: the copies of
# its cells are not always 0
SINGLE = ("inletbody2d", (2, 2))


@pytest.mark.parametrize("deck,shape", M.DECKS)
@pytest.mark.parametrize("prec", ["f64", "f16"])
def test_form_of_the_several_steps_decks(monkeypatch, deck, shape, prec):
    a, b = M._pair(monkeypatch, M._deck(deck), M.PRECS[prec], shape)
    f = a.step_form()
    assert (f["steps_per_pass"] == 1) == (deck in SINGLE), f
    assert f["steps_per_pass"] % 2 == 1 and (f["window"] is None) == (deck in SINGLE)
    assert b.step_form()["steps_per_pass"] == 1
    a.close()
    b.close()


@pytest.mark.parametrize("n,prec,window", [((900, 225), "f32", (64, 32)), ((900, 225), "f16", (64, 32)),
                                           ((2999, 301), "f32", (64, 32)), ((3601, 1003), "f16", (64, 64)),
                                           ((3601, 1003), "bf16", (64, 64)), ((300, 90), "f64", (32, 16)),
                                           ((300, 90), "bf16sr", (32, 32))])
def test_form_of_the_large_windows(monkeypatch, n, prec, window):
    a, b = M._pair(monkeypatch, M._deck(n), M.PRECS[prec])
    assert a.step_form()["steps_per_pass"] >= 3 and b.step_form()["steps_per_pass"] == 1
    assert a.step_form()["window"] == window
    a.close()
    b.close()


@pytest.mark.parametrize("deck,shape", D.DECKS_2D)
@pytest.mark.parametrize("prec", list(D.PRECS))
def test_form_of_the_two_steps_decks(monkeypatch, deck, shape, prec):
    a, b = D._pair(monkeypatch, D._deck(deck), D.PRECS[prec], shape)
    assert a.step_form()["steps_per_pass"] == 2 and b.step_form()["steps_per_pass"] == 1
    assert a.step_form()["row_cells"] % 64 == 0
    a.close()
    b.close()


@pytest.mark.parametrize("prec", ["f64", "f32", "f16"])
def test_form_of_the_ensemble(monkeypatch, prec):
    from imexlb.ensemble import Batch, cylinder_cases
    decks = [M._deck(n) for n in ((28, 24), (61, 20), (150, 60), (90, 33))] + cylinder_cases(3, seed=2)
    for multi, more, steps in (("1", [], True), ("0", [], False), ("1", [M._deck("inletbody2d")], False)):
        monkeypatch.setenv("IMEXLB_MULTI", multi)
        b = Batch(decks + more, precision=M.PRECS[prec])
        f = b.step_form()
        assert (f["steps_per_pass"] >= 3) == steps and (f["windows"] > len(decks)) == steps, f
        b.close()


# the whole lattice in one window, along one axis or both
@pytest.mark.parametrize("n", [(12, 13), (15, 15), (14, 40), (40, 15)])
@pytest.mark.parametrize("prec", ["f64", "f32", "f16"])
def test_one_window_equals_single_steps(monkeypatch, n, prec):
    a, b = M._pair(monkeypatch, M._deck(n), M.PRECS[prec])
    assert a.step_form()["steps_per_pass"] >= 3
    for k in (4, 9, 60):
        a.advance(k)
        b.advance(k)
        M._same(a, b)
    a.close()
    b.close()


@pytest.fixture
def single_steps(monkeypatch):
    monkeypatch.setenv("IMEXLB_MULTI", "0")
    monkeypatch.setenv("IMEXLB_DOUBLE", "0")
    lat = I.Lattice(2, 48, 24, 0, device=0)
    lat.set_params(1.7, 1.0, 0.05)
    lat.set_geometry(12.0, 3.0)
    assert lat.step_form() == {"steps_per_pass": 1, "window": None, "row_cells": 51}
    lat.close()


def test_single_steps_graph_replay(single_steps, r_vec):
    P.test_graph_replay_matches_oracle(r_vec)
    P.test_deferred_phase_steps_match_oracle(r_vec)


@pytest.mark.parametrize("remap", ["0", "1", "3"])
def test_single_steps_block_order(single_steps, remap, r_vec, monkeypatch):
    P.test_block_order_does_not_change_results(remap, r_vec, monkeypatch)


@pytest.mark.parametrize("small_cells", ["0", str(1 << 30)])
def test_single_steps_small_form(single_steps, small_cells, r_vec, monkeypatch):
    P.test_small_lattice_mode_does_not_change_results(small_cells, r_vec, monkeypatch)


@pytest.mark.parametrize("nx,ny,precision", [(2048, 512, I.F64), (4096, 1024, I.F16_F32)])
def test_single_steps_midsize_small_form(single_steps, nx, ny, precision, r_vec, monkeypatch):
    P.test_midsize_lattices_small_form_bitwise(nx, ny, precision, r_vec, monkeypatch)


@pytest.mark.parametrize("block,cpt,persist", [(64, 1, 0), (256, 2, 1), (512, 4, 0), (128, 4, 1), (256, 1, 0)])
def test_single_steps_batch_shapes(single_steps, block, cpt, persist, r_vec):
    B.test_batch_matches_single_lattices(block, cpt, persist, r_vec)


def test_single_steps_ensemble96(single_steps, r_vec):
    C.test_ensemble96_matches_oracle(r_vec)


def test_int64_slot_tables_keep_single_steps(monkeypatch, r_vec):
    """(Only lattices whose populations 32 bits do not address have them.)"""
    monkeypatch.setenv("IMEXLB_SLOTS64", "1")
    for small in (None, "0"):
        if small is not None:
            monkeypatch.setenv("IMEXLB_SMALL_CELLS", small)
        lat, o, _ = P._run_pair("tiny2d", r_vec, 0)
        assert lat.step_form()["steps_per_pass"] == 1
        lat.advance(41)
        o.run(0, 40, 0)
        P.assert_state_equal(lat, o)
        lat.close()
        o.close()
