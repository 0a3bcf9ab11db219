"""FP64 solves of matrices inside larger ones: rows apart by more than their columns, first elements off the vectors'
alignment, NaN all round, at the column classes of the Gram and product kernels.  Reference and tolerances as in
test_gpu_narrow.py and test_gpu_tiles.py: float64 torch, 1e-12, and 2^-23 and 2^-21 more for float32 S and factors."""
import pytest
import torch

import pyloworder_amd as pl

pytestmark = pytest.mark.gpu


def _inside(m, n, dtype, pad, first, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    buf = torch.full((m + 1, first + n + pad), float("nan"), device="cuda", dtype=dtype)
    A = buf[:m, first:first + n]
    A.copy_(torch.randn((m, n), generator=g, device="cuda", dtype=dtype)
            + 3.0 * torch.randn((m, 1), generator=g, device="cuda", dtype=dtype))
    assert A.stride(0) != n and A.data_ptr() == buf.data_ptr() + first * buf.element_size()
    return A


def _check(A, center, dtype):
    Y = A.double()
    if center:
        Y = Y - Y.mean(1, keepdim=True)
    if center == 2:
        Y = Y / (Y * Y).mean(1, keepdim=True)
    U, S, V = (t.double() for t in pl.math.tsqr_svd(A, center=center))
    f4 = dtype == torch.float32
    if Y.shape[0] <= 8192:  # beyond, orthonormal factors that give Y back have its singular values
        So = torch.linalg.svdvals(Y.cpu())
        assert float((S.cpu() - So).norm() / So.norm()) <= 1e-12 + (2.0 ** -23 if f4 else 0.0)
    assert float(((U * S) @ V - Y).norm() / Y.norm()) <= 1e-12 + (2.0 ** -21 if f4 else 0.0)
    for G in (V @ V.t().contiguous(), U.t().contiguous() @ U):
        assert float((G - torch.eye(G.shape[0], device="cuda", dtype=torch.float64)).abs().max()) \
            <= 1e-12 + (2.0 ** -21 if f4 else 0.0)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("pad,first", [(4, 0), (2, 0), (1, 0), (3, 1), (2, 2)])
@pytest.mark.parametrize("n", [8, 16, 30, 32, 48, 64, 65, 96, 130, 160, 224, 256, 300])
def test_svd_inside_a_matrix(n, pad, first, dtype):
    for center in (0, 1, 2):
        _check(_inside(1037 + n, n, dtype, pad, first, n + pad), center, dtype)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("k,n", [(7, 5), (30, 30), (64, 48), (100, 130), (128, 64), (160, 200), (257, 16)])
@pytest.mark.parametrize("pad,first", [(4, 0), (1, 0), (3, 1)])
def test_products_inside_a_matrix(k, n, pad, first, dtype):
    A, X, B = (_inside(r, c, dtype, pad, first, s) for r, c, s in ((2100, k, 1), (2100, n, 2), (k, n, 3)))
    S = torch.rand(k, device="cuda", dtype=dtype) + 0.5
    eps = 2.0 ** -24 if dtype == torch.float32 else 0.0
    for got, ref, terms in ((pl.POD.reconstruct(A, S, B), (A.double() * S.double()) @ B.double(), k),
                            (pl.POD.project(A, X), A.double().t().contiguous() @ X.double(), 2100)):
        assert float((got.double() - ref).norm() / ref.norm()) <= 2 * ((terms + 2) * terms ** 0.5 * 2.0 ** -53 + eps)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("center", [0, 1, 2])
@pytest.mark.parametrize("n", [130, 300])
def test_tall_products_in_a_solve(n, center, dtype):
    """Rows from 2^17 on: 64-row tiles of the U pass, and beyond 256 columns of Z = Y W1 with its zero blocks skipped."""
    _check(_inside((1 << 17) + 65, n, dtype, 3, 1, n), center, dtype)
