"""Narrow FP64 solves at the row counts from which a lone problem's Grams take more chunks: the factors against the
input itself and against orthonormality.  Tolerances as in test_gpu_narrow.py: 1e-12, 2^-21 more for float32 factors."""
import pytest
import torch

import pyloworder_amd as pl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32, torch.complex128])
@pytest.mark.parametrize("m,n", [(1 << 18, 16), ((1 << 18) + 1, 15), (1 << 21, 4), ((1 << 21) + 33, 7)])
def test_svd(m, n, dtype):
    g = torch.Generator(device="cuda").manual_seed(n)
    A = torch.randn((m, n), generator=g, device="cuda", dtype=dtype)
    wide = torch.complex128 if dtype.is_complex else torch.float64
    tol = 1e-12 + (2.0 ** -21 if dtype == torch.float32 else 0.0)
    U, S, V = (t.to(wide) for t in pl.math.tsqr_svd(A))
    assert float(((U * S) @ V - A.to(wide)).norm() / A.to(wide).norm()) <= tol
    assert float((U.conj().t().contiguous() @ U - torch.eye(n, device="cuda", dtype=wide)).norm()) <= n * tol
