"""GPU parity of slk_sddmm_strips (dW over strips).

Every strip size x parts combination gives the oracle's SIMD-order bits, and
the bits of slk_sddmm_bias for dbias, where it can go wrong: row counts that
fill neither a quad nor a workgroup, columns at and around one block, N below a
step, with and without the 8-wide and scalar tails, at and around one window of
either size, N not a multiple of 4 and unaligned dY, rows that are empty, full
(several strips per block) and of mixed length in one quad, padding slots,
values that are not finite, a row order with rows left to the dense kernel.
Bar: bit-exact.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from helpers import assert_bits_equal, from_oracle
from sparsecore_amd import _lib, ops

pytestmark = pytest.mark.gpu

SIZES = [(s, r, v) for s, r in ((48, 1), (32, 1), (16, 1), (16, 2)) for v in (1, 2)]


def _t(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def _mixed(M, K, seed):
    rng = np.random.default_rng(seed)
    W = rng.standard_normal((M, K)).astype(np.float32)
    keep = np.array([0.05, 0.6, 1.0, 0.0, 0.3])[np.arange(M) % 5]
    W *= rng.random((M, K)) < keep[:, None]
    return oracle.from_dense(W)


def _run(W, sizes, dY, X, first=0, ordered=False):
    view = W._view()
    T = _lib.strip_build(view, first, ordered, *sizes, dY.device)
    dW = torch.full((W.total_capacity,), float("nan"), device=dY.device)
    db = torch.full((W.nrows,), float("nan"), device=dY.device)
    _lib.sddmm_strips(view, T, dY, X, dW, db)
    return dW, db


@pytest.mark.parametrize("slots,per_wave,parts", SIZES)
@pytest.mark.parametrize("block", [16, 48, 144])
@pytest.mark.parametrize("M,K,N", [(1, 1, 1), (63, 47, 15), (66, 49, 16), (130, 145, 63),
                                   (70, 150, 64), (257, 96, 130), (65, 300, 251), (64, 144, 264)])
def test_strip_dw_bit_exact(dev, slots, per_wave, parts, block, M, K, N):
    print(f"[strip] {M}x{K} N={N} block={block} {slots}x{per_wave}x{parts}", flush=True)
    c = _mixed(M, K, seed=M + K + N)
    rng = np.random.default_rng(M * N)
    dY_np = rng.standard_normal((M, N)).astype(np.float32)
    X_np = rng.standard_normal((K, N)).astype(np.float32)
    W, dY, X = from_oracle(c, dev), _t(dY_np, dev), _t(X_np, dev)
    want = oracle.sddmm(c, dY_np, X_np, "simd")
    dW, db = _run(W, (block, slots, per_wave, parts), dY, X)
    assert_bits_equal(dW.cpu().numpy(), want, "dW")
    ref, db_ref = torch.empty_like(dW), torch.empty_like(db)
    _lib.sddmm(W._view(), dY, X, ref, _lib.SLK_DW_SIMD, db_ref)
    assert_bits_equal(db.cpu().numpy(), db_ref.cpu().numpy(), "dbias")
    shifted = torch.empty(M * N + 1, device=dev)[1:].view(M, N)
    shifted.copy_(dY)
    dW, _ = _run(W, (block, slots, per_wave, parts), shifted, X)
    assert_bits_equal(dW.cpu().numpy(), want, "unaligned dY")


def test_strip_dw_at_the_largest_block(dev):
    c = _mixed(90, 600, seed=3)
    rng = np.random.default_rng(4)
    dY_np = rng.standard_normal((90, 200)).astype(np.float32)
    X_np = rng.standard_normal((600, 200)).astype(np.float32)
    dW, _ = _run(from_oracle(c, dev), (256, 16, 2, 1), _t(dY_np, dev), _t(X_np, dev))
    assert_bits_equal(dW.cpu().numpy(), oracle.sddmm(c, dY_np, X_np, "simd"), "dW")


@pytest.mark.parametrize("N", [40, 77])
def test_strip_dw_keeps_non_finite_values(dev, N):
    """A slot's dot product takes only its own rows: values that are not finite
    in the columns past the last whole step, or in rows that only padding
    reads, stay out of every other slot."""
    c = _mixed(70, 100, seed=5)
    rng = np.random.default_rng(6)
    dY_np = rng.standard_normal((70, N)).astype(np.float32)
    X_np = rng.standard_normal((100, N)).astype(np.float32)
    X_np[0, :], X_np[7, N - 1], X_np[9, 3], dY_np[5, 2] = np.nan, np.inf, -np.inf, np.inf
    W, dY, X = from_oracle(c, dev), _t(dY_np, dev), _t(X_np, dev)
    want = torch.empty(W.total_capacity, device=dev)
    _lib.sddmm(W._view(), dY, X, want, _lib.SLK_DW_SIMD, None)
    for parts in (1, 2):
        dW, _ = _run(W, (48, 32, 1, parts), dY, X)
        a, b = dW.cpu().numpy(), want.cpu().numpy()
        assert np.array_equal(np.isnan(a), np.isnan(b)) and np.isfinite(b).any()
        assert_bits_equal(np.nan_to_num(a), np.nan_to_num(b), "dW")


def test_strips_of_ordered_rows_leave_the_first_alone(dev):
    c = oracle.zipf_rows(2100, 300, 0.05, 1.1, seed=7, sigma=1.0)
    W = from_oracle(c, dev)
    rng = np.random.default_rng(8)
    dY = _t(rng.standard_normal((2100, 100)).astype(np.float32), dev)
    X = _t(rng.standard_normal((300, 100)).astype(np.float32), dev)
    assert W._view().row_order is not None
    order = W._order[1].cpu().numpy()
    want = torch.empty(W.total_capacity, device=dev)
    _lib.sddmm(W._view(), dY, X, want, _lib.SLK_DW_SIMD, None)
    dW, _ = _run(W, (64, 16, 2, 2), dY, X, first=37, ordered=True)
    got, ref = dW.cpu().numpy(), want.cpu().numpy().copy()
    for r in order[:37]:
        ref[c.row_start[r]:c.row_start[r] + c.row_nnz[r]] = np.nan
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert_bits_equal(np.nan_to_num(got), np.nan_to_num(ref), "dW")


def test_default_route_takes_strips_and_follows_the_topology(dev):
    """Through the autograd path: an odd N takes strips, equal to slk_sddmm, and
    a rewritten row gets new ones."""
    c = oracle.uniform_rows(1200, 500, 200, seed=9, sigma=1.0)
    W = from_oracle(c, dev)
    rng = np.random.default_rng(10)
    X = _t(rng.standard_normal((500, 1001)).astype(np.float32), dev)
    dY = _t(rng.standard_normal((1200, 1001)).astype(np.float32), dev)
    assert ops._strip_sizes(W, 1001) is not None
    for step in range(2):
        dW = ops._launch_sddmm(W, dY, X, "simd")
        want = torch.empty_like(dW)
        _lib.sddmm(W._view(), dY, X, want, _lib.SLK_DW_SIMD, None)
        assert_bits_equal(dW.cpu().numpy(), want.cpu().numpy(), f"dW, step {step}")
        W.rewrite_row(3, list(range(0, 200, 2)), [1.0] * 100)


def test_strips_built_under_capture_stay_with_the_graph(dev, monkeypatch):
    """A first dW under graph capture records choice, build and launch; replays,
    with eager work between them, give the eager bits, and the matrix keeps no
    arrays that only the graph fills."""
    monkeypatch.setitem(ops._overrides, "strips", (144, 48, 1, 2))  # over 64 KiB of LDS
    c = _mixed(200, 300, seed=11)
    W = from_oracle(c, dev)
    rng = np.random.default_rng(12)
    X = _t(rng.standard_normal((300, 129)).astype(np.float32), dev)
    dY = _t(rng.standard_normal((200, 129)).astype(np.float32), dev)
    W._view()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        ops._launch_sddmm(from_oracle(c, dev), dY, X, "simd")  # warm-up on another matrix
        with torch.cuda.graph(graph, stream=stream):
            dW = ops._launch_sddmm(W, dY, X, "simd")
    torch.cuda.current_stream().wait_stream(stream)
    assert not W._strips_kept[1]
    for step in range(3):
        dY.mul_(1.5)
        graph.replay()
        torch.cuda.synchronize()
        assert_bits_equal(dW.cpu().numpy(), ops._launch_sddmm(W, dY, X, "simd").cpu().numpy(),
                          f"replay {step}")
