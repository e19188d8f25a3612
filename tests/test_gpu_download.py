"""Fields downloaded dense, in runs and by several threads, against the
reference's layout (whole padded arrays on one thread): the same values."""
import numpy as np
import pytest

import imexlb as I
from imexlb import _lib

pytestmark = pytest.mark.gpu

# fewer values than a run, a run's and a thread's edges, many runs; 3D
SIZES = [(30, 20, 0), (255, 127, 0), (256, 128, 0), (511, 191, 0), (512, 192, 0), (1023, 511, 0), (1501, 701, 0),
         (24, 17, 13), (127, 63, 47), (150, 120, 60)]


@pytest.mark.parametrize("n", SIZES)
def test_dense_download_equals_reference_layout(n):
    nx, ny, nz = n
    dia = 0.2 * (min(ny, nz) if nz else ny)
    deck = I.Deck(3 if nz else 2, n, dia / nx, 0.3, 50.0, 1.0 / (3.0 * 0.05 * dia / 50.0 + 0.5), 1.0, 1.0, 1.0, 0.01)
    lat, _ = I.setup(deck, np.random.default_rng(9).random(100), device=0)
    for steps in (0, 3, 8):
        lat.advance(steps)
        p, u = lat.download_fields()
        pr, ur = lat.download_fields(_lib.LAYOUT_REF)
        shape = [v + 7 for v in n if v][::-1]
        inner = tuple(slice(3, -3) for _ in shape)
        assert np.array_equal(p, pr.reshape(shape)[inner].ravel())
        ur = ur.reshape(shape + [len(shape)])
        for d in range(len(shape)):
            assert np.array_equal(u[d * lat.N:(d + 1) * lat.N], ur[inner + (d,)].ravel())
    lat.close()
