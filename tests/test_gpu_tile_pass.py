"""The tile pass (block widths up to 16): column counts on both sides of every
tile-height bound, row counts that end inside a tile or before the first,
odd leading dimensions and bases without 16-byte alignment, and columns
beside the ones a product reads.  Against the CPU oracle through the C ABI.

Tolerances: kappa = 1e2, so R and Q agree with the oracle's within a few
n u kappa (n <= 272: 2 * 272 * 1.1e-16 * 1e2 = 6e-12), i.e. 1e-11.
"""
import numpy as np
import pytest

import bcgs_hip as B
import inputs as I
import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

TOL = 1e-11


def run(variant, X, s, ld, shift):
    """Factor X on the device with leading dimension ld, `shift` doubles after
    an allocation's start; pad rows and the surroundings are NaN and must stay.
    Returns Q, R and the status."""
    m, n = X.shape
    buf = torch.full((n * ld + shift + 64,), float("nan"), dtype=torch.float64, device="cuda")
    V = buf[shift:shift + n * ld].view(n, ld)
    V[:, :m] = torch.from_numpy(np.ascontiguousarray(X.T)).cuda()
    R = torch.zeros((n, n), dtype=torch.float64, device="cuda")
    B.bcgs_device(variant, m, n, s, V.data_ptr(), ld, R.data_ptr(), n)
    st = B.status()
    assert torch.isnan(V[:, m:]).all() and torch.isnan(buf[:shift]).all()
    assert torch.isnan(buf[shift + n * ld:]).all()
    return V[:, :m].cpu().numpy().T, R.cpu().numpy().T, st


@pytest.mark.parametrize("variant", ["bcgsi2P1s", "bcgsi21s", "bcgspipi2", "bcgsi2"])
@pytest.mark.parametrize("n,s", [(16, 4), (32, 8), (33, 3), (61, 4), (64, 16), (65, 10), (97, 16),
                                 (128, 8), (129, 16), (144, 10), (200, 10), (256, 16), (257, 16),
                                 (272, 16)])
def test_widths_and_layouts(variant, n, s):
    for m, pad, shift in [(2 * n + 7, 0, 0), (1024 + 32, 0, 0), (3001, 1, 0), (2 * n + 16, 6, 1),
                          (70016 + 129, 3, 2)]:
        if n > 144 and m > 70000:
            continue  # the oracle's time
        print("case tile pass", variant, n, s, m, pad, shift, flush=True)
        X = I.svd_matrix(m, n, 1e2, seed=61)
        Qg, Rg, st = run(variant, X, s, m + pad, shift)
        Qo, Ro, info = O.bcgs(variant, X, s)
        assert st["info_block"] == 0 and info == (0, 0)
        assert np.abs(Rg - Ro).max() <= TOL * np.abs(Ro).max()
        assert np.abs(Qg - Qo).max() <= TOL


@pytest.mark.parametrize("variant", ["bcgsi2P1s", "bcgsi21s", "bcgspipi2"])
@pytest.mark.parametrize("s", [4, 8, 10, 16])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_a_bad_last_block_stays_there(variant, s, bad):
    """One non-finite entry in the last block leaves the blocks before it as
    they are without it: no product of theirs reads its columns."""
    print("case bad last block", variant, s, bad, flush=True)
    n, m = 5 * s, 2000
    X = I.svd_matrix(m, n, 1e2, seed=62)
    _, R0, _ = run(variant, X, s, m, 0)
    X[m // 2, n - 1] = bad
    Q, R, _ = run(variant, X, s, m, 0)
    assert np.array_equal(R[:, :4 * s], R0[:, :4 * s])
    assert np.isfinite(Q[:, :4 * s]).all()
    assert not np.isfinite(R[:, 4 * s:]).all()
