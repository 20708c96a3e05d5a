"""Consecutive calls of the batched form for one batch: a direct run, a capture
with a replay, replays.  Every call sees its own inputs (restored before it)
and gives the same bits as the first, which agrees with the CPU oracle
(kappa = 1e2: within a few n u kappa = 2 * 128 * 1.1e-16 * 1e2 = 2.8e-12, i.e.
1e-11)."""
import numpy as np
import pytest

import bcgs_hip as B
import inputs as I
import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SHAPES = [(4096, 64, 16), (5001, 32, 8), (20000, 128, 16), (4099, 33, 4), (7000, 96, 32),
          (4500, 61, 5)]


@pytest.mark.parametrize("variant", ["bcgsi2P1s", "bcgsi2"])
def test_consecutive_calls_agree(variant):
    print("case batched calls", variant, flush=True)
    ms, ns, ss = zip(*SHAPES)
    hosts = [I.svd_matrix(m, n, 1e2, seed=40 + i) for i, (m, n, s) in enumerate(SHAPES)]
    X0 = [torch.from_numpy(np.ascontiguousarray(h.T)).cuda() for h in hosts]
    X = [torch.empty_like(x) for x in X0]
    R = [torch.zeros((n, n), dtype=torch.float64, device="cuda") for n in ns]
    first = None
    for call in range(5):
        for x, x0, r in zip(X, X0, R):
            x.copy_(x0)
            r.fill_(7.0)
        torch.cuda.synchronize()
        info, _ = B.bcgs_batched_device(variant, ms, ns, ss, [x.data_ptr() for x in X], ms,
                                        [r.data_ptr() for r in R], ns)
        assert all(tuple(i) == (0, 0) for i in info)
        if first is None:
            first = ([x.clone() for x in X], [r.clone() for r in R])
            continue
        assert all(torch.equal(x, f) for x, f in zip(X, first[0])), call
        assert all(torch.equal(r, f) for r, f in zip(R, first[1])), call
    for h, q, r, (m, n, s) in zip(hosts, first[0], first[1], SHAPES):
        Qo, Ro, o = O.bcgs(variant, h, s)
        assert o == (0, 0)
        Rg = np.triu(r.cpu().numpy().T)
        assert np.abs(Rg - np.triu(Ro)).max() <= 1e-11 * np.abs(Ro).max()
        assert np.abs(q.cpu().numpy().T - Qo).max() <= 1e-11
