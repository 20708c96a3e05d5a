"""The tile pass at its widest slabs (block widths up to 8, 273 to 288
columns), where the intra-block QR of the last blocks pads its projection past
the slab's end, and the first slab past them.  Against the CPU oracle.

Tolerance: kappa = 1e2, so R and Q agree with the oracle's within a few
n u kappa (n <= 289: 2 * 289 * 1.1e-16 * 1e2 = 6.4e-12), i.e. 1e-11.
"""
import numpy as np
import pytest

import bcgs_hip as B
import inputs as I
import oracle as O

pytestmark = pytest.mark.gpu

TOL = 1e-11


@pytest.mark.parametrize("variant", list(B.VARIANTS))
@pytest.mark.parametrize("n,s", [(274, 1), (273, 3), (288, 3), (287, 4), (288, 4), (279, 5),
                                 (288, 7), (274, 8), (281, 8), (287, 8), (288, 8), (289, 8)])
def test_widest_slabs(variant, n, s):
    print("case tile pass edge", variant, n, s, flush=True)
    X = I.svd_matrix(1000, n, 1e2, seed=63)
    Qg, Rg, st = B.bcgs(variant, X, s)
    Qo, Ro, info = O.bcgs(variant, X, s)
    assert st["info_block"] == 0 and info == (0, 0)
    assert np.abs(Rg - Ro).max() <= TOL * np.abs(Ro).max()
    assert np.abs(Qg - Qo).max() <= TOL
