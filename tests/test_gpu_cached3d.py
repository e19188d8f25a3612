"""D3Q27 lattices that stay in the caches store their outputs through them;
IMEXLB_SMALL_CELLS=0 takes the streaming stores of larger ones: the same bits,
also against the oracle (which the small decks of the other tests cover)."""
import numpy as np
import pytest

import imexlb as I

pytestmark = pytest.mark.gpu
PRECS = {"f64": I.F64, "f32": I.F32, "f16": I.F16_F32, "bf16": I.BF16_F32, "bf16sr": I.BF16SR_F32}


@pytest.mark.parametrize("n", [(7, 5, 6), (62, 17, 19), (90, 40, 31)])
@pytest.mark.parametrize("prec", list(PRECS))
def test_cached_and_streaming_stores_agree(monkeypatch, n, prec):
    dia = 0.3 * min(n[1:])
    deck = I.Deck(3, n, dia / n[0], 0.3, 50.0, 1.0 / (3.0 * 0.05 * dia / 50.0 + 0.5), 1.0, 1.0, 1.0, 0.01)
    out = []
    for cells in (None, "0"):
        if cells is None:
            monkeypatch.delenv("IMEXLB_SMALL_CELLS", raising=False)
        else:
            monkeypatch.setenv("IMEXLB_SMALL_CELLS", cells)
        lat, _ = I.setup(deck, np.random.default_rng(2).random(100), device=0, precision=PRECS[prec])
        res = []
        for k in (1, 2, 40):
            lat.advance(k)
            res += [lat.download_pdf(I.PDF_F), lat.download_pdf(I.PDF_FB), *lat.download_fields(), lat.forces()]
        out.append(res)
        lat.close()
    for x, y in zip(*out):
        assert np.array_equal(x, y)
