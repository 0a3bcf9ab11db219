"""Real block Jacobi at the edges of its blocks: one pair of 16-column blocks (n <=
32), an odd number of blocks, a ragged last block, the widest single-launch step
(512) and the first two-launch one, clustered and repeated singular values, and
scales whose squares come near the ends of the float64 range.

Tolerance: the passes and the rotations are backward stable, so U S V reproduces A to
a modest multiple of n 2^-53 relative to |A|; 1e-12 holds that for n <= 560 with room.
"""
import numpy as np
import pytest
import torch

import pyloworder_amd as pl

pytestmark = pytest.mark.gpu


def _check(A, tol=1e-12):
    U, S, V = pl.math.tsqr_svd(A)
    n = A.shape[1]
    So = torch.linalg.svdvals(A.cpu())
    eye = torch.eye(n, device="cuda", dtype=torch.float64)
    assert float((S.cpu() - So).norm() / So.norm()) <= tol
    assert bool((S[:-1] >= S[1:]).all())
    assert float(((U * S) @ V - A).norm() / A.norm()) <= tol
    assert float((U.t().contiguous() @ U - eye).abs().max()) <= tol
    assert float((V @ V.t().contiguous() - eye).abs().max()) <= tol


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 32, 33, 48, 49, 64, 95, 129, 255, 300, 511, 512, 513, 545])
def test_block_edges(n):
    g = torch.Generator(device="cuda").manual_seed(n)
    A = torch.randn((2 * n + 100, n), generator=g, device="cuda", dtype=torch.float64)
    _check(A * torch.logspace(0, -4, n, device="cuda", dtype=torch.float64))


@pytest.mark.parametrize("n", [20, 100])
@pytest.mark.parametrize("kind", ["equal", "pairs", "huge", "tiny"])
def test_spectra_and_scales(n, kind):
    g = np.random.default_rng(n)
    Q1, Q2 = np.linalg.qr(g.standard_normal((400, n)))[0], np.linalg.qr(g.standard_normal((n, n)))[0]
    s = {"equal": np.ones(n), "pairs": np.repeat(np.linspace(1, 2, n // 2), 2), "huge": 1e120 * np.linspace(1, 2, n),
         "tiny": 1e-120 * np.linspace(1, 2, n)}[kind]
    _check(torch.from_numpy((Q1 * s) @ Q2.T).cuda())
