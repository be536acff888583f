"""Kept schedules across streams and under graph capture, on the device: a
second stream's first call while the build still waits on the first one, and
replays after warm-up, other sizes and a rewritten row. Bar: the bits of the
same call on a matrix of its own."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from helpers import assert_bits_equal, from_oracle
from sparsecore_amd import layout, ops

pytestmark = pytest.mark.gpu


def _t(shape, dev, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    return torch.randn(shape, generator=g, device=dev)


# quads and strips below 2048 rows; a row order with quads; segment list; phase
# bounds over a skewed matrix with dense rows
CASES = {
    "quads_strips": (1152, 384, 0.3, 1001, "uniform"),
    "order_segments": (2304, 768, 0.1, 2048, "uniform"),
    "dense_rows": (2560, 8256, 0.04, 4160, "zipf"),
}


def _matrix(M, K, d, rows):
    make = oracle.zipf_rows if rows == "zipf" else None
    if make is not None:
        return make(M, K, d, 1.1, seed=3, sigma=1.0)
    return oracle.uniform_rows(M, K, int(d * K), seed=3, sigma=1.0)


@pytest.mark.parametrize("case", list(CASES))
def test_second_stream_waits_for_the_first_ones_build(dev, case):
    M, K, d, N, rows = CASES[case]
    print(f"[two streams] {case} {M}x{K} N={N}", flush=True)
    c = _matrix(M, K, d, rows)
    X, dY = _t((K, N), dev, 1), _t((M, N), dev, 2)
    own = from_oracle(c, dev)
    want = [ops._launch_spmm(own, X), ops._launch_sddmm(own, dY, X, "simd")]
    W = from_oracle(c, dev)
    layout.PaddedCSR._rows_host(W)  # (the row order's host read, before the race)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(a):
        torch.cuda._sleep(int(5e7))  # the builds stay queued behind it
        first = [ops._launch_spmm(W, X), ops._launch_sddmm(W, dY, X, "simd")]
    with torch.cuda.stream(b):
        second = [ops._launch_spmm(W, X), ops._launch_sddmm(W, dY, X, "simd")]
    torch.cuda.synchronize()
    for got in (first, second):
        for g, w, name in zip(got, want, ("Y", "dW")):
            assert_bits_equal(g.cpu().numpy(), w.cpu().numpy(), name)


@pytest.mark.parametrize("forced", [True, False])
@pytest.mark.parametrize("M", [1152, 2304])
def test_replay_after_warm_up_other_sizes_and_a_rewritten_row(dev, monkeypatch, M, forced):
    """Forward and strips' dW follow a row rewritten in place, with quads and
    strips recorded (forced) and by the default rule."""
    K, N = 384, 260 if forced else 1024
    print(f"[capture] {M}x{K} N={N} forced={forced}", flush=True)
    if forced:
        monkeypatch.setitem(ops._overrides, "quad", 1)
        monkeypatch.setitem(ops._overrides, "strips", (48, 32, 1, 2))
    c = oracle.uniform_rows(M, K, 115, seed=4, sigma=1.0)
    W = from_oracle(c, dev)
    X, dY = _t((K, N), dev, 5), _t((M, N), dev, 6)
    run = lambda W, X, dY: [ops._launch_spmm(W, X)] + \
        ([ops._launch_sddmm(W, dY, X, "simd")] if forced else [])
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(3):
            run(W, X, dY)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = run(W, X, dY)
    for n in (64, 100, 333, 1001, 2000, 4096):  # eager, other sizes
        run(W, _t((K, n), dev, n), _t((M, n), dev, n + 1))
    for step in range(3):
        graph.replay()
        torch.cuda.synchronize()
        fresh = layout.PaddedCSR(M, K, W.values, W.col_indices, W.row_start, W.row_nnz,
                                 W.row_capacity)
        for g, w in zip(outs, run(fresh, X, dY)):
            assert_bits_equal(g.cpu().numpy(), w.cpu().numpy(), f"replay {step}")
        n = 115 - 20 * step
        W.rewrite_row(7 + step, list(range(step, step + n)), np.full(n, 0.5, np.float32))
        run(W, X, dY)


def test_captured_input_gradient_keeps_its_transposes_quads(dev, monkeypatch):
    """dX captured after warm-up runs on the quads kept with the cached transpose,
    and replays right after eager calls of other sizes; once the matrix has a new
    topology, a replay still reads the pinned ones (old rows, new values)."""
    monkeypatch.setitem(ops._overrides, "quad", 1)
    c = oracle.uniform_rows(300, 270, 40, seed=7, sigma=1.0)
    W = from_oracle(c, dev)
    X, dY = _t((270, 100), dev, 8), _t((300, 100), dev, 9)
    run = lambda n=None: ops._spmm_backward(W, X, dY if n is None else _t((300, n), dev, n),
                                            "simd", False, True)[1]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(3):
            run()
    torch.cuda.current_stream().wait_stream(side)
    WT = ops._transpose_entry(W)[0]
    assert WT._has("_quads_kept", (1, True))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        dX = run()
    assert len(WT._pinned[1]) == 1 and W._pinned[1][0][2] is WT
    for step in range(3):
        for n in (64, 333, 1001):
            run(n)
        W.values.mul_(-2.0)
        graph.replay()
        torch.cuda.synchronize()
        want = run()
        assert_bits_equal(dX.cpu().numpy(), want.cpu().numpy(), f"replay {step}")
    del WT
    W.rewrite_row(0, [1, 2], [0.0, 0.0])
    assert ops._transpose_entry(W)[0] is not W._pinned[1][0][2]
    torch.empty(1 << 22, device=dev).fill_(float("nan"))
    graph.replay()
    torch.cuda.synchronize()
    assert torch.isfinite(dX).all()
