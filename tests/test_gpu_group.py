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
