"""Tiled FP64 kernels (Grams of 65 to 256 columns and beyond, products over more than
128 inputs) at the edges of their tiles, column classes, K chunks and column slices,
against torch in float64.  Tolerances as in test_gpu_narrow.py: (K + 2) sqrt(K) 2^-53
for a product over K terms, 2^-24 more for float32 results.
"""
import numpy as np
import pytest
import torch

import pyloworder_amd as pl

pytestmark = pytest.mark.gpu


def _rand(m, n, dtype, pad, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn((m, n + pad), generator=g, device="cuda", dtype=dtype)[:, :n]


def _err(a, b):
    return float((a.double() - b).norm() / b.norm())


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("k,n", [(129, 1), (151, 151), (160, 256), (161, 257), (192, 64), (223, 300), (256, 16),
                                 (257, 100), (300, 513), (530, 47)])
def test_tiled_products(k, n, dtype):
    tol = (k + 2) * np.sqrt(k) * 2.0 ** -53 + (2.0 ** -24 if dtype == torch.float32 else 0.0)
    for m in (1024, 4127):
        A, B = _rand(m, k, dtype, 1, 1), _rand(k, n, dtype, 0, 2)
        assert _err(pl.math.matmul(A, B), A.double() @ B.double()) <= tol


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("m,n", [(300, 65), (1000, 96), (1055, 97), (600, 129), (2049, 160), (4000, 161), (777, 193),
                                 (20001, 225), (513, 256), (900, 257), (1500, 385)])
@pytest.mark.parametrize("center", [0, 1, 2])
def test_tiled_svd(m, n, center, dtype):
    A = _rand(m, n, dtype, 3, 5) + 3.0 * _rand(m, 1, dtype, 0, 6)
    Y = A.double()
    if center:
        Y = Y - Y.mean(1, keepdim=True)
    if center == 2:
        Y = Y / (Y * Y).mean(1, keepdim=True)
    U, S, V = pl.math.tsqr_svd(A, center=center)
    So = torch.linalg.svdvals(Y.cpu())
    assert _err(S.cpu(), So) <= 1e-12 + (2.0 ** -23 if dtype == torch.float32 else 0.0)
    assert _err((U.double() * S.double()) @ V.double(), Y) <= 1e-12 + (2.0 ** -21 if dtype == torch.float32 else 0.0)
