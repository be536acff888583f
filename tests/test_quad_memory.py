"""Quads and strips are schedules that slk_spmm and slk_sddmm do without: a call
that cannot have their memory runs on those (no device; the launches are
recorded stand-ins)."""

from __future__ import annotations

import pytest
import torch

import oracle
from helpers import from_oracle
from sparsecore_amd import _lib, layout, ops


@pytest.fixture
def calls(monkeypatch):
    log = []

    def refuse(*a, **k):
        log.append("refused")
        raise torch.OutOfMemoryError("no memory")

    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(_lib, "quad_build", refuse)
    monkeypatch.setattr(_lib, "strip_build", refuse)
    monkeypatch.setattr(_lib, "spmm", lambda v, X, Y, bias=None: log.append(("spmm", v.nrows, bias)))
    monkeypatch.setattr(_lib, "sddmm", lambda v, dY, X, dW, order, db: log.append(("sddmm", db)))
    monkeypatch.setattr(_lib, "transpose_refresh", lambda *a: log.append("refresh"))
    monkeypatch.setattr(_lib, "seg_list_build",
                        lambda v, b, s, dev: [torch.zeros(1, dtype=torch.int32)] * 4)
    monkeypatch.setattr(layout, "_Built", lambda value, arrays: None)
    monkeypatch.setitem(ops._overrides, "fused_backward", False)
    monkeypatch.setitem(ops._overrides, "quad", 1)
    monkeypatch.setitem(ops._overrides, "strips", (48, 32, 1, 2))
    return log


def test_forward_dw_and_dx_run_without_schedules(calls, monkeypatch):
    W = from_oracle(oracle.uniform_rows(40, 30, 9, seed=1))
    WT = from_oracle(oracle.uniform_rows(30, 40, 12, seed=1))
    monkeypatch.setattr(ops, "_transpose_entry", lambda w: (WT, None, False))
    X, dY, b = torch.zeros(30, 8), torch.zeros(40, 8), torch.zeros(40)
    ops._launch_spmm(W, X, b)
    assert calls == ["refused", ("spmm", 40, b)]
    calls.clear()
    dW, dX = ops._spmm_backward(W, X, dY, "simd", True, True, b)
    assert calls == ["refused", ("sddmm", b), "refused", "refresh", ("spmm", 30, None)]
    assert dW.shape == (W.total_capacity,) and dX.shape == (30, 8)
    assert not W._quads_kept[1] and not W._strips_kept[1] and not WT._quads_kept[1]


def test_a_refused_value_buffer_gives_the_kept_quads_up(calls, monkeypatch):
    W = from_oracle(oracle.uniform_rows(40, 30, 9, seed=1))
    monkeypatch.setattr(layout.PaddedCSR, "_quads", lambda *a: object())
    monkeypatch.setattr(_lib, "spmm_quad", _lib.quad_build)
    W._quads_kept = (W.topology_version, {(1, False): "kept"})
    ops._launch_spmm(W, torch.zeros(30, 8))
    assert calls == ["refused", ("spmm", 40, None)] and not W._quads_kept[1]


def test_large_quads_are_not_recorded_in_graphs(monkeypatch):
    v = _lib.CsrView(200000, 4096, int(1.2 * 0.05 * 200000 * 4096), 8, 8, 8, 8, 8)
    assert _lib.quad_halves(v, 8192) > 0 and _lib.quad_bytes(v, 1) > _lib.QUAD_READ_BYTES
    small = _lib.CsrView(2304, 768, int(1.2 * 0.3 * 2304 * 768), 8, 8, 8, 8, 8)
    assert _lib.quad_bytes(small, 1) < _lib.QUAD_READ_BYTES
    W = from_oracle(oracle.uniform_rows(16, 16, 2, seed=1))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    monkeypatch.setattr(layout.PaddedCSR, "nnz", property(lambda W: 1 << 24))
    monkeypatch.setattr(layout.PaddedCSR, "_skewed", lambda W: False)
    for view, takes in ((v, 0), (small, 2)):
        view.routes = {}
        monkeypatch.setattr(layout.PaddedCSR, "_view", lambda W: view)
        assert ops._quad_halves(W, view.ncols, 8192) == takes
