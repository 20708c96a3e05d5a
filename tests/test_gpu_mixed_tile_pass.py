"""The mixed form with FP64 products on the tile pass: tile heights from 16 to
128 rows, the raw FP32 columns in one or two blocks, row counts that end
inside a tile or a group of four rows, and FP32 inputs with and without
16-byte alignment.  Against the CPU oracle on the rounded input.

Tolerances: kappa = 1e2, so R and Q agree with the oracle's within a few
n u kappa (n <= 256: 2 * 256 * 1.1e-16 * 1e2 = 5.7e-12), i.e. 1e-11.
"""
import numpy as np
import pytest

import bcgs_hip as B
import inputs as I
import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

TOL = 1e-11


@pytest.mark.parametrize("m,n", [(128 * 512 + 77, 32), (64 * 512 + 3, 64), (32 * 512 + 32, 128),
                                 (3001, 16), (2000, 144), (1027, 256)])
@pytest.mark.parametrize("pad32,padq,shift", [(0, 0, 0), (3, 2, 1), (5, 1, 0)])
def test_heights_and_layouts(m, n, pad32, padq, shift):
    print("case mixed tile pass", m, n, pad32, padq, shift, flush=True)
    X = I.svd_matrix(m, n, 1e2, seed=81).astype(np.float32)
    ldx, ldq = m + pad32, m + padq
    xb = torch.full((n * ldx + shift,), float("nan"), dtype=torch.float32, device="cuda")
    V = xb[shift:].view(n, ldx)
    V[:, :m] = torch.from_numpy(np.ascontiguousarray(X.T)).cuda()
    Q = torch.full((n, ldq), float("nan"), dtype=torch.float64, device="cuda")
    R = torch.zeros((n, n), dtype=torch.float64, device="cuda")
    B.bcgs_mixed_device("bcgsi2P1s", "fp64", m, n, 16, V.data_ptr(), ldx, Q.data_ptr(), ldq,
                        R.data_ptr(), n)
    assert B.status()["info_block"] == 0
    assert torch.isnan(Q[:, m:]).all()
    Qo, Ro, info = O.bcgs("bcgsi2P1s", np.asfortranarray(X.astype(np.float64)), 16)
    assert info == (0, 0)
    assert np.abs(R.cpu().numpy().T - Ro).max() <= TOL * np.abs(Ro).max()
    assert np.abs(Q[:, :m].cpu().numpy().T - Qo).max() <= TOL
