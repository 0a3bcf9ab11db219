"""Non-finite input is refused with LinAlgError at every size of the small stage, and
the context works on afterwards.  (The pivoted Cholesky completes its permutation with
every index it did not pivot, NaN diagonals included: the permutation addresses rows.)
"""
import numpy as np
import pytest

import pyloworder_amd as pl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [8, 33, 65, 200])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_nonfinite_input_is_refused(n, bad, precision):
    rng = np.random.default_rng(n)
    A = rng.standard_normal((500, n)).astype(np.float32)
    B = A.copy()
    B[123, n // 2] = bad
    with pytest.raises(pl.LinAlgError):
        pl.math.tsqr_svd(B, precision=precision)
    U, S, V = pl.math.tsqr_svd(A, precision=precision)
    assert np.linalg.norm((U * S) @ V - A) <= 1e-5 * np.linalg.norm(A)
