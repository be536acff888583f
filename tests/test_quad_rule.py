"""slk_quad_halves, the rule that sends an SpMM to the row quads, and the host
checks of their entry points (no device)."""

from __future__ import annotations

import ctypes

import pytest

from sparsecore_amd import _lib


def _view(M, K, density, **kw):
    # slot pointers that no host code reads
    return _lib.CsrView(M, K, int(1.2 * density * M * K), 8, 8, 8, 8, 8, **kw)


@pytest.mark.parametrize("M,K,N,density,takes", [
    # measured us, slk_spmm against quads
    (2304, 768, 8192, 0.2, True),     # 219, 169
    (768, 3072, 4096, 0.3, True),     # 265, 169
    (3072, 768, 1001, 0.1, True),     # 82, 35
    (2304, 768, 1024, 0.3, True),     # 70, 51
    (4096, 4096, 4095, 0.01, True),   # 305, 174
    (16384, 4096, 2048, 0.03, True),  # 575, 389
    (2304, 768, 512, 0.1, False),     # 19, 26
    (4096, 4096, 128, 0.1, False),    # 70, 99
    (512, 784, 2048, 0.1, False),     # 16, 24
    (768, 2304, 333, 0.1, False),     # 29, 66
    (256, 256, 8192, 0.3, False),     # 20, 22
    (16384, 4096, 2048, 0.01, False),  # 240, 288
    (3072, 768, 8, 0.1, False),
])
def test_quads_only_where_they_measured_faster(M, K, N, density, takes):
    assert (_lib.quad_halves(_view(M, K, density), N) > 0) == takes


def test_quads_leave_skewed_dense_and_forced_matrices_alone(tune):
    M, K, N, d = 2304, 768, 8192, 0.2
    assert _lib.quad_halves(_view(M, K, d), N) == 2
    assert _lib.quad_halves(_view(M, K, d, n_heavy_rows=1), N) == 0
    assert _lib.quad_halves(_view(M, K, d, n_dense_rows=32), N) == 0
    assert _lib.quad_halves(_view(M, K, d), 3) == 0
    assert _lib.quad_halves(_view(M, K, d), (1 << 22) + 1) == 0
    assert _lib.quad_halves(_view(0, K, d), N) == _lib.quad_halves(_view(M, 0, d), N) == 0
    for knob in ("spmm_kernel", "spmm_h", "spmm_rw", "spmm_split", "spmm_vec", "spmm_bin", "spmm_g",
                 "dense_rows"):
        tune(**{knob: 0})
        assert _lib.quad_halves(_view(M, K, d), N) == 0, knob
        _lib.set_tuning(knob, None)


def test_quad_entry_points_check_their_arguments():
    lib = _lib.load()
    v = _view(8, 300, 0.1)
    ref = ctypes.byref(v)
    assert lib.slk_quad_chunks(300, 1) == 2 and lib.slk_quad_chunks(300, 2) == 3
    assert lib.slk_quad_chunks(300, 3) == lib.slk_quad_chunks(0, 1) == 0
    n = lib.slk_quad_windows(ref, 1)
    assert n == v.total_capacity // 16 + 2 * 2
    rc = lib.slk_quad_build(ref, None, 3, 8, 24, 8, 8, 8, 8, n, 8, None)
    assert rc == _lib.SLK_EINVAL and "halves" in lib.slk_last_error().decode()
    rc = lib.slk_quad_build(ref, None, 1, 8, 23, 8, 8, 8, 8, n, 8, None)
    assert rc == _lib.SLK_EINVAL and "workspace" in lib.slk_last_error().decode()
    rc = lib.slk_quad_build(ref, None, 1, 8, 24, 8, 8, 8, 8, n - 1, 8, None)
    assert rc == _lib.SLK_EINVAL and "workspace" in lib.slk_last_error().decode()
    rc = lib.slk_quad_build(ref, None, 1, 8, 24, None, 8, 8, 8, n, 8, None)
    assert rc == _lib.SLK_EINVAL and "NULL" in lib.slk_last_error().decode()
    q = _lib.QuadView(8, 8, 8, 8, 8, n, 1)
    call = lambda Q, K, N: lib.slk_spmm_quad(ref, ctypes.byref(Q), 8, 8, 8, K, N, None, 8, None)
    assert call(_lib.QuadView(), 300, 8) == _lib.SLK_EINVAL
    assert call(q, 299, 8) == _lib.SLK_EINVAL and "shape" in lib.slk_last_error().decode()
    assert call(q, 300, 3) == _lib.SLK_EINVAL and "N outside" in lib.slk_last_error().decode()


def test_more_windows_than_their_scan_counts_are_refused():
    lib = _lib.load()
    v = _lib.CsrView(1 << 26, 65536, 31 << 26, 8, 8, 8, 8, 8)
    assert lib.slk_quad_windows(ctypes.byref(v), 1) > 2 ** 31
    assert _lib.quad_halves(v, 4095) == 0
    rc = lib.slk_quad_count(ctypes.byref(v), 1, 8, 1 << 40, 8, 8, 8, None)
    assert rc == _lib.SLK_EINVAL and "windows" in lib.slk_last_error().decode()
    rc = lib.slk_quad_fill(ctypes.byref(v), None, 1, 8, 1 << 40, 8, 8, 8, 8, 64, 8, None)
    assert rc == _lib.SLK_EINVAL and "windows" in lib.slk_last_error().decode()
