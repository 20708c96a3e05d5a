"""Inputs scaled towards the ends of the exponent range, where the Gram's
entries (and a Cholesky pivot's reciprocal) leave the normal range but the
factors do not: X 2^e, whose Q is X's and whose R is X's times 2^e.

Tolerances: at e = -520 the Gram keeps 1074 - 1040 = 34 bits (kappa = 1e2, so
its error is 2^-34 kappa^2 = 6e-7 of its smallest eigenvalue); the second
normalization, at unit scale, brings orthogonality to a few n u (n <= 96: 10 n
u = 1e-13) in all variants but A-1S, whose last normalization is that Gram's.
R is formed from the factors that were applied, so the residual stays at a few
u: 1e-14.
"""
import numpy as np
import pytest

import bcgs_hip as B
import inputs as I

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", list(B.VARIANTS))
@pytest.mark.parametrize("s", [4, 10, 16, 32])
@pytest.mark.parametrize("e", [-520, -512, 500, 506])
def test_scaled_input(variant, s, e):
    n, m = 3 * s, 1500
    X0 = I.svd_matrix(m, n, 1e2, seed=8)
    print("case scaled input", variant, s, e, flush=True)
    Q, R, st = B.bcgs(variant, np.asfortranarray(np.ldexp(X0, e)), s)
    assert st["info_block"] == 0
    R = np.ldexp(R, -e)
    assert np.linalg.norm(Q @ R - X0) <= 1e-14 * np.linalg.norm(X0)
    if variant != "bcgsi21s":
        assert I.loo(Q) <= 1e-13
