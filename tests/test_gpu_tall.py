"""Products around the row count from which a workgroup takes 64-row tiles: the last rows of a tile, column blocks that
leave waves idle, inputs in one and in two chunks.  FP64 sums of at most 300 terms of order one, 1e-12 of the largest."""
import pytest
import torch

import pyloworder_amd as pl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [(1 << 17) - 1, 1 << 17, (1 << 17) + 65])
@pytest.mark.parametrize("k,n", [(130, 129), (160, 256), (256, 200), (300, 270)])
def test_reconstruct(m, k, n):
    g = torch.Generator(device="cuda").manual_seed(m + k)
    U = torch.randn((m, k), generator=g, device="cuda", dtype=torch.float64)
    S = torch.rand(k, generator=g, device="cuda", dtype=torch.float64) + 0.5
    V = torch.randn((k, n), generator=g, device="cuda", dtype=torch.float64)
    ref = (U * S) @ V
    out = pl.POD.reconstruct(U, S, V)
    assert float((out - ref).abs().max()) <= 1e-12 * float(ref.abs().max())
