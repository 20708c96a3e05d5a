"""The wide-block pass with one slice of the inner dimension (up to 256 buffer
columns): a group's second Z tile is subtracted in place only after every wave
has read the group's columns, which the folded schedules' second group
multiplies.  Widths whose written columns lie in the unit of 16 columns that
step 1 reads last (19, 21 to 23, 25 to 31) and in the one it reads first (17,
20, 24, 32); 16-, 32- and 64-row tiles.

A column read after the subtraction would leave a residual of about u kappa
(1e-11 at kappa = 1e5) and results that differ between runs.  Bound: the
residual of a factorization by normalized blocks is a few u (u = 1.1e-16) per
pass over a column, below 1e-14 for two passes; repeats agree bit for bit
(every sum has a fixed order).
"""
import pytest

import bcgs_hip as B
import device_inputs as D

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("variant", ["bcgsi2P1s", "bcgsi2P2s", "bcgsi21s"])
@pytest.mark.parametrize("s", [17, 19, 20, 21, 22, 23, 24, 25, 26, 27, 28, 29, 30, 31, 32])
def test_residual_and_repeat(variant, s):
    for n in sorted({2 * s, 64, 128 // s * s, 128, 250 // s * s, 251, 256}):
        m = 70001
        print("case wide pass handover", variant, n, s, flush=True)
        X0 = D.svd_input(torch, m, n, 1e5, seed=91 + s)
        out = []
        for _ in range(2):
            X = X0.clone()
            R = torch.zeros((n, n), dtype=torch.float64, device="cuda")
            B.bcgs_device(variant, m, n, s, X.data_ptr(), m, R.data_ptr(), n)
            assert B.status()["info_block"] == 0
            out.append((X, R))
        (X, R), (X2, R2) = out
        _, res, xn = B.accuracy_device(m, n, X0.data_ptr(), m, X.data_ptr(), m, R.data_ptr(), n)
        assert res <= 1e-14 * xn, (n, s, res / xn)
        assert torch.equal(X, X2) and torch.equal(R, R2), (n, s)
