"""Dense factorisations of the small stage (k_dense.hip) at the edges of their panels, lane columns and size
classes, through the solves that run them.  A = Q diag(s) V^T has exact singular values; the FP64 solve's error
is a small multiple of n u times the largest one (1e-13 n gives it 40 times n u sigma_1 of room at any n here)."""
import numpy as np
import pytest
import torch

import pyloworder_amd as pl

pytestmark = pytest.mark.gpu
EDGES = [1, 2, 3, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 192, 193, 255, 256, 257, 320, 384, 385, 511, 512,
         513]


def _orth(rng, m, n):
    return np.linalg.qr(rng.standard_normal((m, n)))[0]


@pytest.mark.parametrize("n", EDGES)
@pytest.mark.parametrize("rank", ["full", "half"])
def test_factor_sizes(n, rank):
    rng = np.random.default_rng(n)
    m, k = 2 * n + 40, n if rank == "full" else (n + 1) // 2
    s = np.linspace(2.0, 1.0, k)
    A = (_orth(rng, m, k) * s) @ _orth(rng, n, k).T
    U, S, VT = (x.cpu().numpy() for x in pl.math.tsqr_svd(torch.from_numpy(A).cuda()))
    tol = 1e-13 * max(n, 10)
    assert np.abs(S[:k] - s).max() <= tol and (k == n or S[k:].max() <= tol)
    assert np.abs((U * S) @ VT - A).max() <= tol
    assert np.abs(U.T @ U - np.eye(n)).max() <= tol and np.abs(VT @ VT.T - np.eye(n)).max() <= tol
    Q, R = (x.cpu().numpy() for x in pl.math.tsqr(torch.from_numpy(A).cuda()))
    assert np.abs(Q @ R - A).max() <= tol and np.abs(Q.T @ Q - np.eye(n)).max() <= tol


@pytest.mark.parametrize("n", [33, 64, 200, 300])
def test_equal_diagonals(n):
    """An orthonormal input: every pivot of the second factorisation ties with the others up to rounding."""
    Q = _orth(np.random.default_rng(7), 4 * n, n)
    U, S, VT = (x.cpu().numpy() for x in pl.math.tsqr_svd(torch.from_numpy(Q).cuda()))
    assert np.abs(S - 1).max() <= 1e-13 * n and np.abs((U * S) @ VT - Q).max() <= 1e-13 * n


@pytest.mark.parametrize("n,r", [(256, 74), (200, 17), (64, 33)])
def test_restarted_shift(n, r):
    """Sketches after power steps are so ill-conditioned that the shifted factorisation restarts with a larger
    shift, some pivots in: the result is orthonormal and holds A's leading part all the same."""
    rng = np.random.default_rng(r)
    s = 1e3 * 0.8 ** np.arange(n)
    A = (_orth(rng, 4 * n, n) * s) @ _orth(rng, n, n).T
    U, S, VT = (x.cpu().numpy() for x in pl.math.randomized_svd(torch.from_numpy(A).cuda(), r, 3, seed=5))
    assert np.abs(U.T @ U - np.eye(r)).max() <= 1e-13 * n
    # three power steps and a gap of 0.8 per mode: what is lost is far below the first mode left out's energy
    assert np.linalg.norm(A - (U * S) @ VT, 2) <= 2 * s[r]


@pytest.mark.parametrize("n", [1, 2, 3, 5, 12, 31, 64, 65, 72, 73, 100])
@pytest.mark.parametrize("kind", ["random", "rotations"])
def test_eig_sizes(n, kind):
    """Eigenpairs by their residual (n u ||A|| of the backward-stable QR iteration, with room) and trace; below and
    above one lane per column and the size whose arrays fit in LDS. Rotations: every eigenvalue in a pair of modulus 1
    (and one 1), none of which the iteration may split into reals."""
    rng = np.random.default_rng(n)
    A = rng.standard_normal((n, n))
    if kind == "rotations":
        Q = _orth(rng, n, n)
        th = np.linspace(0.3, 2.8, n // 2)
        D = np.eye(n)
        for i, t in enumerate(th):
            D[2 * i:2 * i + 2, 2 * i:2 * i + 2] = [[np.cos(t), -np.sin(t)], [np.sin(t), np.cos(t)]]
        A = Q @ D @ Q.T
    wr, wi, V = (x.cpu().numpy() for x in pl.math.eigen(torch.from_numpy(A).cuda()))
    w = wr + 1j * wi
    tol = 1e-13 * max(n, 10) * np.linalg.norm(A, 2)
    assert np.abs(A @ V - V * w).max() <= tol
    assert abs(w.sum() - np.trace(A)) <= tol * n
    assert np.abs(np.linalg.norm(V, axis=0) - 1).max() <= 1e-13
    if kind == "rotations":
        assert np.abs(np.abs(w) - 1).max() <= tol and (np.abs(wi) > 0.1).sum() == 2 * (n // 2)


@pytest.mark.parametrize("missing", [1, 2, 4, 5])
@pytest.mark.parametrize("dtype", [np.float64, np.complex128])
def test_few_null_directions(missing, dtype):
    """Completion of U where a wave forms each sum (up to four directions) and where a thread does."""
    rng = np.random.default_rng(missing)
    n, m = 40, 300
    k = n - missing

    def orth(r, c):
        z = rng.standard_normal((r, c)) + (1j * rng.standard_normal((r, c)) if dtype is np.complex128 else 0)
        return np.linalg.qr(z)[0]

    s = np.linspace(2.0, 1.0, k)
    A = (orth(m, k) * s) @ orth(n, k).conj().T
    U, S, VT = (x.cpu().numpy() for x in pl.math.tsqr_svd(torch.from_numpy(A).cuda()))
    tol = 1e-13 * n
    assert np.abs(S[:k] - s).max() <= tol and S[k:].max() <= tol
    assert np.abs(U.conj().T @ U - np.eye(n)).max() <= tol and np.abs((U * S) @ VT - A).max() <= tol


@pytest.mark.parametrize("dtype,n", [(np.float64, 142), (np.float64, 143), (np.float64, 180), (np.float64, 181),
                                     (np.complex128, 100), (np.complex128, 101), (np.complex128, 181)])
def test_qr_signs_at_the_forms_of_their_factorisation(dtype, n):
    """R and Q as numpy.linalg.qr, signs and all, where the shifted LU leaves LDS and where its rows go to waves: 1e-9
    of max |R|, 1e-8 for Q, as in test_tsqr_lapack_signs."""
    rng = np.random.default_rng(n)
    A = rng.standard_normal((700, n)).astype(dtype)
    if np.iscomplexobj(A):
        A = A + 1j * rng.standard_normal((700, n))
    Q, R = pl.math.tsqr(A)
    Qo, Ro = np.linalg.qr(A)
    assert np.abs(R - Ro).max() <= 1e-9 * np.abs(Ro).max()
    assert np.abs(Q - Qo).max() <= 1e-8
