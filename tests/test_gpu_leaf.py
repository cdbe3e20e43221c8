"""The panel leaf at the edges of its launch shapes: one workgroup up to 512
rows (1 or 2 rows per thread), several above; ties and columns without a
comparable candidate decided as the oracle decides them."""
import numpy as np
import pytest

import lu2_amd as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["gepp", "compat"])
@pytest.mark.parametrize("n,nb", [(256, 32), (288, 32), (512, 64), (544, 32), (1024, 128), (1056, 32), (2080, 32)])
def test_leaf_ties_and_columns_without_candidate(ctx, oracle, n, nb, mode):
    """Pivots exactly the oracle's.  Column 0 holds one magnitude only (the
    lowest row wins a tie); a NaN column from the middle of a leaf on leaves
    no candidate there or, through its update, anywhere behind it (the
    current row stays)."""
    gpu, ref = (L.PIV_GEPP, oracle.PIV_GEPP) if mode == "gepp" else (L.PIV_COMPAT, oracle.PIV_COMPAT)
    a0 = oracle.randomsetmat(n, n + nb)
    a0[:, 0] = np.where(a0[:, 0] < 0, -0.5, 0.5)
    _, piv, _ = L.solve(a0, nb, gpu, ctx)
    _, po, _ = oracle.lumcolumn(a0, nb, ref)
    assert po[0] == 0
    assert np.array_equal(piv, po)
    a0[:, 21] = np.nan
    _, piv, _ = L.solve(a0, nb, gpu, ctx)
    assert np.array_equal(piv[:21], po[:21])
    if mode == "gepp":   # under the odd-column rule column 21 pivots on column 20
        assert np.array_equal(piv[21:], np.arange(21, n))
