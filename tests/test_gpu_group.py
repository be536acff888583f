"""GPU parity of slk_spmm's packed kernel for N < 64 (several rows per wave):
rows of 0 to 49 slots, at and around one and two batches of 16, in one wave;
N at and around each lane width; a last wave that is partly empty; a padded
batch beside values that are not finite. Bar: the oracle's bits."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from helpers import assert_bits_equal, from_oracle
from sparsecore_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 2, 7, 8, 9, 16, 17, 31, 32])
@pytest.mark.parametrize("M", [1, 5, 131])
def test_packed_rows_bit_exact(dev, M, N):
    print(f"[packed] M={M} N={N}", flush=True)
    K = 60
    rng = np.random.default_rng(M + N)
    W = np.zeros((M, K), np.float32)
    for r in range(M):
        n = (16, 0, 1, 15, 17, 32, 33, 31, 49)[r % 9]
        W[r, rng.choice(K - 1, n, replace=False)] = rng.standard_normal(n)
    c = oracle.from_dense(W)
    X = rng.standard_normal((K, N)).astype(np.float32)
    X[K - 1] = np.inf  # a column that no row holds
    b = rng.standard_normal(M).astype(np.float32)
    Wd, Xd = from_oracle(c, dev), torch.from_numpy(X).to(dev)
    Y = torch.full((M, N), float("nan"), device=dev)
    _lib.spmm(Wd._view(), Xd, Y)
    want = oracle.spmm(c, X)
    assert_bits_equal(Y.cpu().numpy(), want, "Y")
    _lib.spmm(Wd._view(), Xd, Y, torch.from_numpy(b).to(dev))
    assert_bits_equal(Y.cpu().numpy(), want + b[:, None], "Y + bias")


@pytest.mark.parametrize("N", [1, 2, 3, 5, 9, 32])
@pytest.mark.parametrize("kind", ["one", "few", "mixed", "zipf", "beside_dense"])
def test_every_row_length_and_order_bit_exact(dev, kind, N):
    """Above 16384 rows with 4 slots or fewer: as many lanes as columns, batches of
    2, 4 and 8; longer and mixed rows; skewed rows, longest first; the rows beside
    dense ones, which only the row order lists."""
    print(f"[packed] {kind} N={N}", flush=True)
    rng = np.random.default_rng(N)
    K = 70
    if kind == "zipf":
        c = oracle.zipf_rows(2100, 300, 0.03, 1.1, seed=N, sigma=1.0)
    elif kind == "beside_dense":
        K = 4096
        lens = [K if r % 60 == 7 else r % 5 for r in range(2100)]
    else:
        M = 16397
        lens = {"one": np.ones(M, int), "few": np.arange(M) % 5,
                "mixed": np.arange(M) // 64 * 3 % 41}[kind]
    if kind != "zipf":
        cols = [np.sort(rng.choice(K, n, replace=False)).astype(np.int32) for n in lens]
        c = oracle.from_row_lists(len(lens), K, cols,
                                  [rng.standard_normal(n).astype(np.float32) for n in lens], 0.2)
    W = from_oracle(c, dev)
    v = W._view()
    assert (v.n_dense_rows > 0) == (kind == "beside_dense")
    if kind == "beside_dense":
        assert v.n_heavy_rows == v.n_dense_rows
    X = rng.standard_normal((c.ncols, N)).astype(np.float32)
    b = rng.standard_normal(c.nrows).astype(np.float32)
    Y = torch.full((c.nrows, N), float("nan"), device=dev)
    _lib.spmm(v, torch.from_numpy(X).to(dev), Y, torch.from_numpy(b).to(dev))
    want = oracle.spmm(c, X) + b[:, None]
    if kind == "beside_dense":  # equal under ==: a dense row's zero may differ in sign
        np.testing.assert_array_equal(Y.cpu().numpy(), want)
    else:
        assert_bits_equal(Y.cpu().numpy(), want, "Y")
