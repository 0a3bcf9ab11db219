"""Members of a group end their Jacobi sweeps at their own test: members that need none, few and many sweeps, in one
block pair and in several, give what a lone solve gives, bit for bit."""
import pytest
import torch

import pyloworder_amd as pl

pytestmark = pytest.mark.gpu


def _member(kind, m, n, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    A = torch.randn((m, n), generator=g, device="cuda", dtype=torch.float64)
    k = torch.arange(n, device="cuda", dtype=torch.float64)
    if kind == "orthogonal":  # unit columns of disjoint rows
        A = torch.zeros_like(A)
        A[torch.arange(m, device="cuda"), torch.arange(m, device="cuda") % n] = 1.0
    elif kind == "graded":
        A *= 0.9 ** k
    elif kind == "mixed up":  # graded in a turned basis: the sweeps have the most to do
        A = (A * 0.8 ** k) @ torch.linalg.qr(torch.randn((n, n), generator=g, device="cuda", dtype=torch.float64))[0]
    elif kind == "constant":
        A[:] = 1.0
    return A.to(dtype)


@pytest.mark.parametrize("dtype,precision", [(torch.float64, "fp64"), (torch.float32, "mixed")])
def test_members_equal_lone_solves(dtype, precision):
    shapes = [(3000, 8), (2500, 33), (4000, 48), (3100, 100), (5000, 129), (2000, 200), (3000, 256)]
    kinds = ["random", "orthogonal", "graded", "mixed up", "constant"]
    As = [_member(k, m, n, dtype, 7 * i + j) for i, (m, n) in enumerate(shapes) for j, k in enumerate(kinds)]
    for A, *usv in zip(As, *pl.math.tsqr_svd_grouped(As, precision=precision)):
        for got, want in zip(usv, pl.math.tsqr_svd(A, precision=precision)):
            assert torch.equal(got, want), tuple(A.shape)
