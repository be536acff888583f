"""GPU parity of slk_spmm_quad (row quads) and of their device builder.

The builder's arrays equal the numpy restatement below entry for entry; the
kernel, forced onto every quads-per-wave x halves variant, gives the oracle's
bits where it can go wrong: row counts that fill neither a quad nor a row
block, K at and around one chunk, N at and around one column tile and not a
multiple of 4, unaligned X, rows that are empty, full (a chunk's largest count
and most windows) and of mixed length in one quad, bias, a transpose read
through its slot map, values changed after the build, zeros of both signs and
values that are not finite (a padded slot must not touch them).
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

CONFIGS = [(1, rw) for rw in (3, 4, 6, 8, 9, 16)] + [(2, rw) for rw in (3, 4, 6, 8)]


@pytest.fixture
def quad(monkeypatch):
    """quad(h) runs every SpMM through quads of h halves, quad(0) none."""
    return lambda h: monkeypatch.setitem(ops._overrides, "quad", h)


def _t(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def _mixed(M, K, seed):
    """Rows 0%, 5%, 60% and 100% dense in turn: every quad mixes them."""
    rng = np.random.default_rng(seed)
    W = rng.standard_normal((M, K)).astype(np.float32)
    keep = np.array([0.05, 0.6, 1.0, 0.0, 0.3])[np.arange(M) % 5]
    W *= rng.random((M, K)) < keep[:, None]
    return oracle.from_dense(W)


def _quads(c, halves):
    """start, count, offset, slot of the definition beside slk_quads."""
    kc = 252 // halves
    nq, nc = -(-c.nrows // 4), -(-c.ncols // kc)
    start, count = np.zeros((nc, nq), np.int32), np.zeros((nc, nq), np.uint8)
    off, slot = [], []
    for q in range(nq):
        for ch in range(nc):
            runs = []
            for r in range(4 * q, 4 * q + 4):
                s = np.arange(c.row_start[r], c.row_start[r] + c.row_nnz[r]) if r < c.nrows else \
                    np.zeros(0, np.int64)
                runs.append(s[(c.col_indices[s] >= ch * kc) & (c.col_indices[s] < (ch + 1) * kc)] if len(s) else s)
            n = max(map(len, runs))
            nw = max(1, -(-n // 16))
            start[ch, q], count[ch, q] = len(off) // 64, n
            o, sl = np.full((nw, 4, 16), 64512, np.int64), np.full((nw, 4, 16), -1, np.int64)
            for r, run in enumerate(runs):
                i = np.arange(len(run))
                o[i // 16, r, i % 16] = (c.col_indices[run] - ch * kc) * 256 * halves
                sl[i // 16, r, i % 16] = run
            off += o.ravel().tolist()
            slot += sl.ravel().tolist()
    return start, count, np.array(off, np.int32), np.array(slot, np.int32)


@pytest.mark.parametrize("halves", [1, 2])
@pytest.mark.parametrize("M,K", [(1, 1), (63, 251), (64, 252), (66, 253), (130, 700)])
def test_quad_build_matches_the_restatement(dev, halves, M, K):
    print(f"[quad build] {M}x{K} halves={halves}", flush=True)
    c = _mixed(M, K, seed=M + K)
    W = from_oracle(c, dev)
    q = W._quads(halves)
    start, count, offset, slot, used = (a.cpu().numpy() for a in q.arrays)
    w_start, w_count, w_off, w_slot = _quads(c, halves)
    n = int(used[-1])
    assert 64 * n == len(w_off) and n <= q.n_windows
    assert_bits_equal(start, w_start.ravel(), "start")
    assert_bits_equal(count, w_count.ravel(), "count")
    assert_bits_equal(offset[:64 * n], w_off, "offset")
    assert_bits_equal(slot[:64 * n], w_slot, "slot")


@pytest.mark.parametrize("halves,rw", CONFIGS)
@pytest.mark.parametrize("M,K,N", [(1, 1, 4), (191, 126, 64), (193, 252, 129), (387, 253, 68),
                                   (1030, 505, 260), (70, 1000, 127)])
def test_quad_spmm_bit_exact(dev, quad, tune, halves, rw, M, K, N):
    quad(halves)
    tune(quad_rw=rw)
    print(f"[quad spmm] {M}x{K} N={N} halves={halves} rw={rw}", flush=True)
    c = _mixed(M, K, seed=M + K + N)
    rng = np.random.default_rng(M + N)
    X_np = rng.standard_normal((K, N)).astype(np.float32)
    b_np = rng.standard_normal(M).astype(np.float32)
    W, X = from_oracle(c, dev), _t(X_np, dev)
    want = oracle.spmm(c, X_np)
    assert_bits_equal(ops._launch_spmm(W, X).cpu().numpy(), want, "Y")
    W.values.mul_(-2.0)  # exact, and after the build
    assert_bits_equal(ops._launch_spmm(W, X, _t(b_np, dev)).cpu().numpy(),
                      -2.0 * want + b_np[:, None], "bias")
    shifted = torch.empty(K * N + 1, device=dev)[1:].view(K, N)
    shifted.copy_(X)
    assert_bits_equal(ops._launch_spmm(W, shifted).cpu().numpy(), 0.0 - 2.0 * want, "unaligned X")


@pytest.mark.parametrize("halves", [1, 2])
@pytest.mark.parametrize("N", [72, 75])
def test_quad_input_gradient_through_the_slot_map(dev, quad, halves, N):
    """dX by quads of the transpose, values read from W: after a change of W's
    values the bits of the refreshed transpose's slk_spmm."""
    c = _mixed(300, 270, seed=N)
    dY = _t(np.random.default_rng(N).standard_normal((300, N)).astype(np.float32), dev)
    X = torch.zeros(270, N, device=dev)
    W = from_oracle(c, dev)
    for step in range(2):
        W.values.add_(0.25)
        quad(halves)
        dX = ops._spmm_backward(W, X, dY, "simd", False, True)[1]
        quad(0)
        want = ops._launch_spmm(ops._cached_transpose(W), dY)
        assert_bits_equal(dX.cpu().numpy(), want.cpu().numpy(), f"dX, step {step}")


@pytest.mark.parametrize("halves", [1, 2])
def test_quad_keeps_signed_zeros_and_non_finite_values(dev, quad, halves):
    c = _mixed(130, 300, seed=7)
    rng = np.random.default_rng(8)
    X_np = rng.standard_normal((300, 68)).astype(np.float32)
    X_np[rng.random(X_np.shape) < 0.3] = -0.0
    X_np[:, 0] = -0.0
    X_np[17, 3], X_np[18, 4], X_np[19, 5] = np.inf, -np.inf, np.nan
    W, X = from_oracle(c, dev), _t(X_np, dev)
    quad(0)
    want = ops._launch_spmm(W, X).cpu().numpy()
    quad(halves)
    got = ops._launch_spmm(W, X).cpu().numpy()
    assert np.isnan(want).any() and np.isinf(want).any()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert_bits_equal(np.nan_to_num(got), np.nan_to_num(want), "Y")


def test_quads_built_under_capture_stay_with_the_graph(dev, quad):
    """A first call under graph capture records the build; replays (with eager
    work between them) give the eager bits, and the matrix keeps no arrays that
    only the graph fills."""
    quad(1)
    c = _mixed(200, 300, seed=9)
    W = from_oracle(c, dev)
    X = _t(np.random.default_rng(9).standard_normal((300, 128)).astype(np.float32), dev)
    W._view()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        ops._launch_spmm(from_oracle(c, dev), X)  # warm-up on another matrix
        with torch.cuda.graph(graph, stream=stream):
            Y = ops._launch_spmm(W, X)
    torch.cuda.current_stream().wait_stream(stream)
    assert not W._quads_kept[1]
    for step in range(3):
        W.values.mul_(1.5)
        graph.replay()
        torch.cuda.synchronize()
        quad(1)
        assert_bits_equal(Y.cpu().numpy(), ops._launch_spmm(W, X).cpu().numpy(), f"replay {step}")


@pytest.mark.parametrize("halves", [1, 2])
@pytest.mark.parametrize("M,K", [(1, 1), (66, 253), (130, 700)])
def test_quads_sized_by_their_count_match_the_bound_sized(dev, monkeypatch, quad, halves, M, K):
    """Above QUAD_READ_BYTES (here: always) offset and slot hold the windows used
    and no more; the arrays, of a matrix and of its transpose, and the product
    are the same."""
    print(f"[quad exact size] {M}x{K} halves={halves}", flush=True)
    c = _mixed(M, K, seed=M + K)
    X = _t(np.random.default_rng(M).standard_normal((K, 68)).astype(np.float32), dev)
    W = from_oracle(c, dev)
    WT, perm, _ = ops._transpose_entry(W)
    bound = [W._quads(halves), WT._quads(halves, perm)]
    monkeypatch.setattr(_lib, "QUAD_READ_BYTES", 0)
    W._quads_kept = WT._quads_kept = (-1, {})
    for b, q in zip(bound, (W._quads(halves), WT._quads(halves, perm))):
        n = int(b.arrays[4][-1])
        assert q.n_windows == n <= b.n_windows
        for i, name in enumerate(("start", "count", "offset", "slot", "used")):
            want = b.arrays[i] if i not in (2, 3) else b.arrays[i][:64 * n]
            assert_bits_equal(q.arrays[i].cpu().numpy(), want.cpu().numpy(), name)
    quad(halves)
    assert_bits_equal(ops._launch_spmm(W, X).cpu().numpy(), oracle.spmm(c, X.cpu().numpy()), "Y")
