"""After a breakdown the columns before the bad pivot stay finite: the blocked
triangular solve of the fused passes does not multiply the entries of the bad
column and those after it into the columns before.  Block widths on both sides
of a 4- and a 16-column block, ragged groups, bad columns at the start, in the
middle and at the end of a block.

A zero column gives an exactly zero pivot in every variant (all its products
are zero); a NaN entry makes every product with its column NaN.
"""
import numpy as np
import pytest

import bcgs_hip as B
import inputs as I

pytestmark = pytest.mark.gpu

WIDTHS = [2, 3, 4, 5, 7, 8, 10, 16, 17, 20, 32]


def run(variant, s, blk, j, entry):
    n, m = 4 * s, 2000 if s < 16 else 3000
    X = I.svd_matrix(m, n, 1e2, seed=7)
    c = blk * s + j
    if entry == 0.0:
        X[:, c] = 0.0
    else:
        X[m // 2 + 5, c] = entry
    Q, R, st = B.bcgs(variant, X, s)
    assert (st["info_block"], st["info_pivot"]) == (blk + 1, j + 1)
    assert not np.isfinite(Q[:, c]).any()
    return Q[:, :c], R[:, :c]


def places(s):
    return sorted({s // 2, s - 1, min(s - 1, 6)})


@pytest.mark.parametrize("variant", list(B.VARIANTS))
@pytest.mark.parametrize("s", WIDTHS)
def test_zero_column_in_the_first_block(variant, s):
    for j in places(s):
        print("case breakdown columns, first block", variant, s, j, flush=True)
        Q, R = run(variant, s, 0, j, 0.0)
        assert np.isfinite(Q).all() and np.isfinite(R).all()


@pytest.mark.parametrize("variant", ["bcgsi21s", "bcgspipi2"])
@pytest.mark.parametrize("s", WIDTHS)
@pytest.mark.parametrize("blk", [2, 3])
@pytest.mark.parametrize("entry", [0.0, float("nan")])
def test_bad_column_in_a_later_block(variant, s, blk, entry):
    """Variants whose passes read no column of the block but its own."""
    for j in places(s):
        print("case breakdown columns", variant, s, blk, j, entry, flush=True)
        Q, _ = run(variant, s, blk, j, entry)
        assert np.isfinite(Q).all()
