"""Field downloads on both sides of the sizes that take a plain copy of the
padded arrays (above 16 KiB of one, below 80 Ki values in all)."""
import numpy as np
import pytest

import imexlb as I
import test_gpu_multi as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(2, 2, 0), (42, 42, 0), (43, 43, 0), (2, 800, 0), (163, 163, 0), (165, 165, 0), (9, 9, 9),
                               (10, 10, 10), (26, 26, 26), (27, 27, 27)])
def test_downloads_equal_the_reference_layout(n):
    print(f"[download] {n}", flush=True)
    dim = 3 if n[2] else 2
    lat = I.Lattice(dim, *n, device=0)
    lat.set_params(1.7, 1.0, 0.05)
    lat.set_geometry(0.5 * n[0], 0.2 * min(n[:dim]))
    lat.init_up(np.linspace(0.0, 1.0, 100))
    lat.init_pdf()
    lat.advance(5)
    p, u = lat.download_fields()
    pr, ur = lat.download_fields(I.LAYOUT_REF)
    ax = [v + 7 for v in n[:dim][::-1]]
    inner = tuple(slice(3, -3) for _ in range(dim))
    pr, ur = pr.reshape(ax)[inner], ur.reshape(*ax, dim)[inner]
    assert np.array_equal(p, pr.ravel())
    for d in range(dim):
        assert np.array_equal(u.reshape(dim, -1)[d], ur[..., d].ravel())
    assert np.abs(u).max() > 0
    lat.close()


def test_small_cases_of_an_ensemble():
    from imexlb.ensemble import Batch
    decks = [M._deck(n) for n in ((28, 24), (61, 50), (150, 60), (200, 160))]
    b = Batch(decks)
    b.init(np.linspace(0.0, 1.0, 100))
    b.advance(9)
    for i, dk in enumerate(decks):
        lat, _ = I.setup(dk, np.linspace(0.0, 1.0, 100), device=0)
        lat.advance(9)
        for x, y in zip(lat.download_fields(), b.download_fields(i)):
            assert np.array_equal(x, y)
        lat.close()
    b.close()
