"""The wide-block pass (block widths 17 to 32): column counts on both sides of
every tile-height and wave-count bound, blocks that end inside a 16-column
tile, row counts that end inside a tile or before the first, odd leading
dimensions and bases without 16-byte alignment, and fixed scratch that holds
fewer row chunks than CUs.  Against the CPU oracle through the C ABI.

Tolerances: kappa = 1e2, so R and Q agree with the oracle's within a few
n u kappa (n <= 512: 2 * 512 * 1.1e-16 * 1e2 = 1.1e-11), i.e. 2e-11.
"""
import numpy as np
import pytest

import bcgs_hip as B
import inputs as I
import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

TOL = 2e-11
VARIANTS = ["bcgsi2P1s", "bcgsi21s", "bcgspipi2", "bcgsi2", "bcgsi2P2s"]


def run(variant, X, s, ld, shift, noalloc=False):
    """Factor X on the device with leading dimension ld, `shift` doubles after
    an allocation's start; pad rows and the surroundings are NaN and must stay.
    Returns Q, R and the first breakdown."""
    m, n = X.shape
    buf = torch.full((n * ld + shift + 64,), float("nan"), dtype=torch.float64, device="cuda")
    V = buf[shift:shift + n * ld].view(n, ld)
    V[:, :m] = torch.from_numpy(np.ascontiguousarray(X.T)).cuda()
    R = torch.zeros((n, n), dtype=torch.float64, device="cuda")
    if noalloc:
        info = torch.zeros(2, dtype=torch.int32, device="cuda")
        assert B.bcgs_device_noalloc(variant, m, n, s, V.data_ptr(), ld, R.data_ptr(), n,
                                     info.data_ptr(), 0) == 0
        torch.cuda.synchronize()
        blk = int(info[0])
    else:
        B.bcgs_device(variant, m, n, s, V.data_ptr(), ld, R.data_ptr(), n)
        blk = B.status()["info_block"]
    assert torch.isnan(V[:, m:]).all() and torch.isnan(buf[:shift]).all()
    assert torch.isnan(buf[shift + n * ld:]).all()
    return V[:, :m].cpu().numpy().T, R.cpu().numpy().T, blk


def check(variant, X, s, ld, shift, noalloc=False):
    Qg, Rg, blk = run(variant, X, s, ld, shift, noalloc)
    Qo, Ro, info = O.bcgs(variant, X, s)
    assert blk == 0 and info == (0, 0)
    assert np.abs(Rg - Ro).max() <= TOL * np.abs(Ro).max()
    assert np.abs(Qg - Qo).max() <= TOL


@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("n,s", [(32, 32), (40, 20), (64, 32), (65, 32), (96, 20), (128, 32),
                                 (129, 17), (160, 32), (250, 25), (256, 32), (257, 32),
                                 (300, 20), (500, 24), (511, 31), (512, 32)])
def test_widths_and_layouts(variant, n, s):
    for m, pad, shift in [(2 * n + 7, 0, 0), (1024 + 32, 0, 0), (2 * n + 16, 6, 1), (3001, 1, 0)]:
        if n > 256 and m > 2000:
            continue  # the oracle's time
        print("case wide pass", variant, n, s, m, pad, shift, flush=True)
        check(variant, I.svd_matrix(m, n, 1e2, seed=71), s, m + pad, shift)


@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("m,n,s,pad", [(32 * 512 + 33, 128, 32, 0), (64 * 512 + 129, 64, 32, 1),
                                       (64 * 512, 100, 25, 0), (64 * 512 + 2, 48, 24, 2)])
def test_tall_tiles(variant, m, n, s, pad):
    """Enough rows for the 32- and 64-row tiles."""
    print("case wide pass tall", variant, m, n, s, flush=True)
    check(variant, I.svd_matrix(m, n, 1e2, seed=72), s, m + pad, 0)


@pytest.mark.parametrize("variant", ["bcgsi2P1s", "bcgsi21s"])
def test_fixed_scratch(variant):
    """512 columns on the fixed scratch, whose partials leave CUs without work."""
    print("case wide pass fixed scratch", variant, flush=True)
    check(variant, I.svd_matrix(4100, 512, 1e2, seed=73), 32, 4100, 0, noalloc=True)


@pytest.mark.parametrize("variant", ["bcgsi2P1s", "bcgsi21s", "bcgspipi2"])
@pytest.mark.parametrize("s", [17, 32])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_a_bad_last_block_stays_there(variant, s, bad):
    """One non-finite entry in the last block leaves the blocks before it as
    they are without it: no product of theirs reads its columns."""
    print("case wide pass bad last block", variant, s, bad, flush=True)
    n, m = 5 * s, 2000
    X = I.svd_matrix(m, n, 1e2, seed=74)
    _, R0, _ = run(variant, X, s, m, 0)
    X[m // 2, n - 1] = bad
    Q, R, _ = run(variant, X, s, m, 0)
    assert np.array_equal(R[:, :4 * s], R0[:, :4 * s])
    assert np.isfinite(Q[:, :4 * s]).all()
    assert not np.isfinite(R[:, 4 * s:]).all()
