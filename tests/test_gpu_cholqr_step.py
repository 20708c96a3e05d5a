"""The CholQR steps of narrow blocks run in workgroups of 256 threads: block
widths on both sides of the line (11), ragged last blocks, and partial counts
from one workgroup up, against the CPU oracle, and bit for bit against the
reduction and the step in launches of their own (one summation order; every
entry of a step is computed in one fixed order whatever the workgroup size).

Tolerance: kappa = 1e2, n <= 60, so R agrees with the oracle's within a few
n u kappa (2 * 60 * 1.1e-16 * 1e2 = 1.3e-12), i.e. 1e-11.
"""
import numpy as np
import pytest

import bcgs_hip as B
import inputs as I
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", ["bcgsi2", "bcgsi2P2s", "bcgsi2P1s"])
@pytest.mark.parametrize("s,n", [(1, 5), (2, 9), (3, 20), (8, 45), (10, 50), (11, 36), (12, 60),
                                 (16, 59), (32, 59)])
@pytest.mark.parametrize("m", [64, 1000, 40001])
def test_narrow_steps(variant, s, n, m, monkeypatch):
    print("case cholqr step", variant, s, n, m, flush=True)
    X = I.svd_matrix(m, n, 1e2, seed=91)
    Q, R, st = B.bcgs(variant, X, s)
    _, Ro, info = O.bcgs(variant, X, s)
    assert st["info_block"] == 0 and info == (0, 0)
    assert np.abs(R - Ro).max() <= 1e-11 * np.abs(Ro).max()
    monkeypatch.setenv("ORTH_SEPARATE_REDUCE", "1")
    Q2, R2, _ = B.bcgs(variant, X, s)
    assert np.array_equal(R, R2) and np.array_equal(Q, Q2)
