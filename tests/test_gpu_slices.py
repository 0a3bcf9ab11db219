"""Products over at most 128 inputs at each way their rows and columns are dealt to workgroups: narrow slices of few
rows, half slices, slices side by side and one after the other, W's staging in one part and in several, odd widths.
Cross products around the numbers of chunks and of entries from which their slabs are summed otherwise.
Tolerances as in test_gpu_narrow.py: (K + 2) sqrt(K) 2^-53 for a product over K terms, 2^-24 more for float32 results.
"""
import numpy as np
import pytest
import torch

import pyloworder_amd as pl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("m,k,n", [(1024, 128, 256), (1100, 37, 19), (5003, 128, 999), (20011, 128, 256), (10007, 64, 131),
                                   (60001, 100, 300), (60001, 101, 203), (70001, 16, 64), (70001, 30, 200),
                                   (65537, 17, 16), (131073, 64, 64)])
def test_products(m, k, n, dtype):
    g = torch.Generator(device="cuda").manual_seed(m)
    A = torch.randn((m, k), generator=g, device="cuda", dtype=dtype)
    B = torch.randn((k, n), generator=g, device="cuda", dtype=dtype)
    ref = A.double() @ B.double()
    tol = (k + 2) * np.sqrt(k) * 2.0 ** -53 + (2.0 ** -24 if dtype == torch.float32 else 0.0)
    for C in (pl.math.matmul(A, B), pl.POD.reconstruct(A, torch.ones(k, device="cuda", dtype=dtype), B)):
        assert float((C.double() - ref).norm() / ref.norm()) <= tol
        assert float((C.double() - ref).abs().max()) <= 8 * tol * float(ref.abs().max())


@pytest.mark.parametrize("m,k,n,dtype", [(1100003, 3, 41, torch.float64), (900001, 30, 60, torch.float64),
                                         (1100003, 13, 67, torch.float32), (700003, 16, 131, torch.float32),
                                         (2200003, 5, 17, torch.float64)])
def test_products_beyond_the_cache(m, k, n, dtype):
    """Results of more than 256 MB, their rows on both sides of a line's length and no multiple of it."""
    g = torch.Generator(device="cuda").manual_seed(n)
    A = torch.randn((m, k), generator=g, device="cuda", dtype=dtype)
    B = torch.randn((k, n), generator=g, device="cuda", dtype=dtype)
    C = pl.math.matmul(A, B)
    tol = (k + 2) * np.sqrt(k) * 2.0 ** -53 + (2.0 ** -24 if dtype == torch.float32 else 0.0)
    for r in range(0, m, 1 << 18):
        ref = A[r:r + (1 << 18)].double() @ B.double()
        assert float((C[r:r + (1 << 18)].double() - ref).norm() / ref.norm()) <= tol


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32, torch.complex128, torch.complex64])
@pytest.mark.parametrize("m,k,n", [(200, 5, 3), (8192, 30, 30), (8193, 30, 30), (8193, 17, 64), (70000, 33, 20),
                                   (9001, 70, 65), (9001, 256, 256), (9001, 257, 256)])
def test_cross_products(m, k, n, dtype):
    g = torch.Generator(device="cuda").manual_seed(m + k)
    A = torch.randn((m, k), generator=g, device="cuda", dtype=dtype)
    B = torch.randn((m, n), generator=g, device="cuda", dtype=dtype)
    wide = torch.complex128 if dtype.is_complex else torch.float64
    ref = A.to(wide).conj().t().contiguous() @ B.to(wide)
    tol = (m + 2) * np.sqrt(m) * 2.0 ** -53 + (2.0 ** -24 if dtype in (torch.float32, torch.complex64) else 0.0)
    assert float((pl.POD.project(A, B).to(wide) - ref).norm() / ref.norm()) <= 2 * tol
