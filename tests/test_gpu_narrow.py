"""Narrow FP64 kernels (Grams and cross products of at most 64 columns, products of
at most 128 inputs) at the edges of their tiles, vectors and alignments, against
torch in float64.

Tolerances: a sum of K products in FP64, in any order, is within (K + 2) 2^-53 of the
sum of the moduli, which for Gaussian data is at most sqrt(K) of the result's size in
the Frobenius norm; float32 outputs add 2^-24.
"""
import numpy as np
import pytest
import torch

import pyloworder_amd as pl

pytestmark = pytest.mark.gpu


def _tol(k, dtype):
    return (k + 2) * np.sqrt(k) * 2.0 ** -53 + (2.0 ** -24 if dtype == torch.float32 else 0.0)


def _err(a, b):
    return float((a.double() - b).norm() / b.norm())


def _rand(m, n, dtype, pad, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn((m, n + pad), generator=g, device="cuda", dtype=dtype)[:, :n]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("k,n,pad", [(1, 1, 0), (16, 17, 3), (30, 30, 2), (33, 48, 0), (64, 64, 0), (64, 256, 1),
                                     (65, 129, 0), (74, 256, 2), (128, 100, 0)])
def test_narrow_products(k, n, pad, dtype):
    for m in (1, 17, 1024, 4111):
        A, B, X = _rand(m, k, dtype, pad, 1), _rand(k, n, dtype, 0, 2), _rand(m, n, dtype, pad, 3)
        S = torch.rand(k, device="cuda", dtype=dtype)
        R = pl.POD.reconstruct(A, S, B)
        assert _err(R, (A.double() * S.double()) @ B.double()) <= 2 * _tol(k, dtype)
        C = pl.POD.project(A, X)
        assert _err(C, A.double().t().contiguous() @ X.double()) <= 2 * _tol(m, dtype)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("m,n", [(16, 16), (129, 15), (1025, 30), (777, 32), (3001, 33), (4099, 48), (131073, 64)])
@pytest.mark.parametrize("center", [0, 1, 2])
def test_narrow_svd(m, n, center, dtype):
    A = _rand(m, n, dtype, 2, 5) + 3.0 * _rand(m, 1, dtype, 0, 6)
    Y = A.double()
    if center:
        Y = Y - Y.mean(1, keepdim=True)
    if center == 2:
        Y = Y / (Y * Y).mean(1, keepdim=True)
    U, S, V = pl.math.tsqr_svd(A, center=center)
    So = torch.linalg.svdvals(Y.cpu())
    assert _err(S.cpu(), So) <= 1e-12 + (2.0 ** -23 if dtype == torch.float32 else 0.0)
    assert _err((U.double() * S.double()) @ V.double(), Y) <= 1e-12 + (2.0 ** -21 if dtype == torch.float32 else 0.0)
