"""The separate projection and update kernels (ORTH_UNFUSED=1) at widths that
run a fused pass by default: the widest wide-block slab, the widest narrow-block
one, and both kinds of update (paired on MFMA, row-wise), beside the fused
passes on the same input.  Against the CPU oracle through the C ABI.

Tolerances: kappa = 1e2, so R and Q agree with the oracle's within a few
n u kappa (n <= 512: 2 * 512 * 1.1e-16 * 1e2 = 1.1e-11), i.e. 2e-11.
"""
import numpy as np
import pytest

import bcgs_hip as B
import inputs as I
import oracle as O

pytestmark = pytest.mark.gpu

TOL = 2e-11


@pytest.mark.parametrize("variant", list(B.VARIANTS))
@pytest.mark.parametrize("m,n,s", [(3000, 512, 32), (2001, 250, 25), (2000, 288, 8), (1501, 61, 4),
                                   (2000, 250, 16)])
def test_separate_kernels_beside_the_fused_passes(variant, m, n, s, monkeypatch):
    X = I.svd_matrix(m, n, 1e2, seed=83)
    Qo, Ro, info = O.bcgs(variant, X, s)
    assert info == (0, 0)
    passes = []
    for env in [(), ("ORTH_UNFUSED",), ("ORTH_UNFUSED", "ORTH_UPDATE_ROWWISE")]:
        for name in env:
            monkeypatch.setenv(name, "1")
        print("case separate kernels", variant, m, n, s, env, flush=True)
        Q, R, st = B.bcgs(variant, X, s)
        assert st["info_block"] == 0
        assert np.abs(R - Ro).max() <= TOL * np.abs(Ro).max()
        assert np.abs(Q - Qo).max() <= TOL
        passes.append(st["passes"])
    assert passes[0] < passes[1] == passes[2]
