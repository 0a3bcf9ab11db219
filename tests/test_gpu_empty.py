"""Products over no rows: a sum of nothing is zero, at every width class of the operands."""
import pytest
import torch

import pyloworder_amd as pl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32, torch.complex128])
@pytest.mark.parametrize("k,n", [(1, 1), (16, 17), (33, 64), (64, 64), (40, 65), (100, 20), (300, 8)])
def test_project_of_no_rows_is_zero(k, n, dtype):
    pl.POD.project(torch.ones((5000, k), device="cuda", dtype=dtype), torch.ones((5000, n), device="cuda", dtype=dtype))
    C = pl.POD.project(torch.empty((0, k), device="cuda", dtype=dtype), torch.empty((0, n), device="cuda", dtype=dtype))
    torch.cuda.synchronize()
    assert C.shape == (k, n) and float(C.abs().max()) == 0.0
    assert pl.POD.reconstruct(torch.empty((0, k), device="cuda", dtype=dtype), torch.ones(k, device="cuda"),
                              torch.ones((k, n), device="cuda", dtype=dtype)).shape == (0, n)
