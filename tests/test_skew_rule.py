"""Which skewed matrices below 2048 rows, whose views count no heavy rows, take
row quads and strips (host only; the matrices live on the CPU)."""

from __future__ import annotations

import pytest
import torch

import oracle
from helpers import from_oracle
from sparsecore_amd import ops


@pytest.fixture(autouse=True)
def eager(monkeypatch):
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)


def _matrix(kind, M, K, d):
    if kind == "uniform":
        return from_oracle(oracle.uniform_rows(M, K, int(d * K), seed=1))
    return from_oracle(oracle.zipf_rows(M, K, d, 1.1, seed=1))


@pytest.mark.parametrize("kind,M,K,d,N,quads,strips", [
    # measured us against slk_spmm and slk_sddmm: (fwd), (dW); - where not taken
    ("zipf", 1024, 2048, 0.10, 8192, False, False),  # 271, 370
    ("zipf", 2000, 4096, 0.10, 8192, False, False),  # 930, 991
    ("zipf", 2000, 4096, 0.03, 2048, False, False),  # -; 94, 207
    ("zipf", 2000, 4096, 0.03, 8192, True, False),   # 795, 593; 394, 740
    ("zipf", 512, 2048, 0.10, 8192, True, False),    # 244, 185; 174, 328
    ("zipf", 2000, 784, 0.10, 1001, True, False),    # 120, 94; 52, 79
    ("zipf", 2000, 2048, 0.10, 4095, True, True),    # 850, 367; 804, 317
    ("uniform", 1024, 2048, 0.10, 8192, True, False),  # 164, 138
    ("uniform", 2000, 4096, 0.03, 2048, False, True),  # -; 132, 84
    ("uniform", 2000, 784, 0.10, 1001, True, True),    # 62, 35; 52, 34
])
def test_skewed_rows_take_quads_and_strips_only_where_faster(kind, M, K, d, N, quads, strips):
    W = _matrix(kind, M, K, d)
    assert (ops._quad_halves(W, K, N) > 0) == quads
    assert (ops._strip_sizes(W, N) is not None) == strips


def test_the_count_follows_a_rewritten_row():
    W = _matrix("uniform", 64, 64, 0.1)
    assert not W._skewed()
    for r in range(0, 64, 16):
        W.rewrite_row(r, [], [])
    assert not W._skewed()
    W = _matrix("uniform", 64, 64, 0.5)
    for r in range(64):
        if r % 8:
            W.rewrite_row(r, [0], [1.0])
    assert W._skewed()
