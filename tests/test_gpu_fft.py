"""Welch blocks by the LDS FFT at every power-of-two length it takes: even and odd powers (a last radix-2 stage), one
row, an odd number of rows, and numbers of blocks that leave the last pass and chunk partly filled.  Float32 transforms
against the oracle's float64 ones, 2e-6 of the largest value times the square root of the blocks as in the SPOD tests."""
import numpy as np
import pytest

import oracle
import pyloworder_amd as pl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ndft", [4, 8, 16, 32, 64, 128, 256, 512, 1024, 2048])
@pytest.mark.parametrize("rows,blocks", [(1, 1), (7, 5), (18, 21)])
def test_lengths(ndft, rows, blocks):
    rng = np.random.default_rng(ndft + rows)
    nolap = ndft // 4
    n = blocks * (ndft - nolap) + nolap
    t = 0.01 * np.arange(n)
    X = (rng.standard_normal((rows, n)) + 50.0).astype(np.float32)
    Qo, fo, nbo = oracle.spod_blocks(X.astype(np.float64), t, ndft, nolap)
    Q, f, nb = pl.SPOD.blocks(X, t, ndft, nolap)
    assert nb == nbo == blocks and np.array_equal(f, fo) and Q.shape == Qo.shape
    assert np.abs(Q - Qo).max() <= 2e-6 * np.abs(Qo).max() * np.sqrt(Qo.shape[2])


@pytest.mark.parametrize("rows,n", [(1, 2), (7, 300), (18, 1024), (5, 1999)])
def test_length_two(rows, n):
    """The shortest transform, y0 +- y1: one block to several chunks of them, same bounds."""
    rng = np.random.default_rng(n)
    t = 0.01 * np.arange(n)
    X = (rng.standard_normal((rows, n)) + 50.0).astype(np.float32)
    Qo, fo, nbo = oracle.spod_blocks(X.astype(np.float64), t, 2, 1)
    Q, f, nb = pl.SPOD.blocks(X, t, 2, 1)
    assert nb == nbo == n - 1 and np.array_equal(f, fo) and Q.shape == Qo.shape
    assert np.abs(Q - Qo).max() <= 2e-6 * np.abs(Qo).max() * np.sqrt(Qo.shape[2])
