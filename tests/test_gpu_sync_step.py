"""The synchronization step (prefix Gram on MFMA tiles, one-wave Cholesky of
the two blocks' joint matrix, R and coefficient tiles) at the widths and
prefixes where its tiles end, and the end of a call (R and status by one
kernel): against the CPU oracle through the C ABI.

Tolerances: at kappa = 1e2 every quantity of the step has a relative error of
a few n u kappa (n <= 132, u = 1.1e-16: 3e-12 for n u kappa * 2), so R and Q
agree with the oracle's within 1e-11.
"""
import numpy as np
import pytest

import bcgs_hip as B
import inputs as I
import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

TOL = 1e-11


@pytest.mark.parametrize("variant", list(B.VARIANTS))
@pytest.mark.parametrize("s,n", [(1, 6), (2, 17), (4, 33), (5, 31), (8, 47), (15, 46), (16, 130),
                                 (16, 33), (17, 52), (24, 121), (31, 93), (32, 65), (32, 132)])
def test_step_widths(variant, s, n):
    """Block widths on both sides of a 16-column tile, ragged last blocks of
    one column up, prefixes that end inside a 16-row tile."""
    print("case step widths", variant, s, n, flush=True)
    m = 40 * n
    X = I.svd_matrix(m, n, 1e2, seed=51)
    Qg, Rg, st = B.bcgs(variant, X, s)
    Qo, Ro, info = O.bcgs(variant, X, s)
    assert st["info_block"] == 0 and info == (0, 0)
    assert np.abs(Rg - Ro).max() <= TOL * np.abs(Ro).max()
    assert np.abs(Qg - Qo).max() <= TOL


@pytest.mark.parametrize("variant", ["bcgsi2P1s", "bcgspipi2"])
@pytest.mark.parametrize("s,n,bad", [(5, 20, 2), (16, 48, 2), (32, 96, 3)])
def test_breakdown_is_reported(variant, s, n, bad):
    """A zero column in block `bad` (1-based) gives a zero pivot there (every
    product with it is exactly zero): the same block and pivot as the oracle,
    and R finite before it."""
    print("case breakdown", variant, s, n, flush=True)
    X = I.svd_matrix(50 * n, n, 1e2, seed=52)
    X[:, (bad - 1) * s + s // 2] = 0.0
    _, R, st = B.bcgs(variant, X, s)
    _, _, info = O.bcgs(variant, X, s)
    assert (st["info_block"], st["info_pivot"]) == info == (bad, s // 2 + 1)
    assert np.isfinite(R[:, :(bad - 1) * s]).all()


@pytest.mark.parametrize("s,n,pad", [(5, 23, 0), (16, 40, 3), (32, 300, 1)])
@pytest.mark.parametrize("where", ["device", "pinned"])
def test_only_block_rows_of_R_are_written(s, n, pad, where):
    """R with a leading dimension above n, in device or pinned host memory:
    rows below each block column and the padding keep their contents."""
    print("case R rows", s, n, where, flush=True)
    m = 20 * n
    X = I.svd_matrix(m, n, 1e2, seed=53)
    dX = torch.from_numpy(np.ascontiguousarray(X.T)).cuda()
    ld = n + pad
    R = torch.full((n, ld), 7.5, dtype=torch.float64)
    R = R.cuda() if where == "device" else R.pin_memory()
    B.bcgs_device("bcgsi2P1s", m, n, s, dX.data_ptr(), m, R.data_ptr(), ld)
    B.sync()
    torch.cuda.synchronize()
    R = R.cpu().numpy().T
    _, Ro, _ = O.bcgs("bcgsi2P1s", X, s)
    for j in range(n):
        end = min(n, (j // s + 1) * s)
        assert np.abs(R[:end, j] - Ro[:end, j]).max() <= TOL * np.abs(Ro).max()
        assert (R[end:, j] == 7.5).all()
