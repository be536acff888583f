"""slk_strip_choose, the rule that sends a weight gradient to the strips, and
the host checks of their entry points (no device)."""

from __future__ import annotations

import ctypes

import pytest

from sparsecore_amd import _lib


def _view(M, K, density, **kw):
    # slot pointers that no host code reads
    return _lib.CsrView(M, K, int(1.2 * density * M * K), 8, 8, 8, 8, 8, **kw)


@pytest.mark.parametrize("M,K,N,density,takes", [
    # measured us, slk_sddmm against strips
    (2304, 768, 8192, 0.3, True),     # 373, 280
    (1152, 384, 8192, 0.2, True),     # 251, 107
    (512, 784, 8192, 0.2, True),      # 159, 108
    (2304, 768, 256, 0.2, True),      # 31, 16
    (4096, 4096, 512, 0.1, True),     # 266, 116
    (4096, 4096, 4096, 0.05, True),   # 585, 380
    (3072, 3072, 4095, 0.1, True),    # 2014, 393
    (1000, 1000, 1000, 0.4, True),    # 110, 43
    (512, 784, 256, 0.1, False),      # 8, 11
    (256, 256, 8192, 0.2, False),     # 60, 81
    (768, 3072, 8192, 0.1, False),    # 216, 226
    (2304, 768, 1024, 0.7, False),    # 98, 104
    (8192, 4096, 2048, 0.1, False),   # 633, 649
    (768, 2304, 333, 0.03, False),    # 10, 21
    (3072, 768, 8, 0.1, False),
])
def test_strips_only_where_they_measured_faster(M, K, N, density, takes):
    assert (_lib.strip_choose(_view(M, K, density), N)[0] is not None) == takes


@pytest.mark.parametrize("M,K,N,density,takes", [
    # measured us, slk_sddmm against strips: where the segment kernel gains, and beside it
    (4096, 4096, 8192, 0.1, False),   # 1254, 1402
    (768, 4096, 1024, 0.05, False),   # 34, 40
    (1000, 768, 1024, 0.1, False),    # 19, 23
    (1537, 1000, 8192, 0.05, False),  # 128, 137
    (4096, 384, 4096, 0.05, True),    # 130, 68
    (256, 784, 8192, 0.25, True),     # 117, 94
    (4096, 2048, 8192, 0.2, True),    # 1115, 983
    (2000, 2048, 2048, 0.03, True),   # 63, 56
])
def test_strips_not_where_the_segment_kernel_gains(M, K, N, density, takes):
    assert (_lib.strip_choose(_view(M, K, density), N)[0] is not None) == takes


def test_strips_leave_skewed_and_dense_rows_alone():
    assert _lib.strip_choose(_view(2304, 768, 0.3), 8192)[0] is not None
    assert _lib.strip_choose(_view(2304, 768, 0.3, row_order=8, n_heavy_rows=1), 8192)[0] is None
    assert _lib.strip_choose(_view(2304, 768, 0.3, row_order=8, n_dense_rows=32, dense_ws=256), 8192)[0] is None
    assert _lib.strip_choose(_view(0, 768, 0.3), 8192)[0] is None
    assert _lib.strip_choose(_view(2304, 768, 0.3), 0)[0] is None
    assert _lib.strip_choose(_view(2304, 768, 0.3), (1 << 21) + 1)[0] is None


def test_strip_entry_points_check_their_arguments():
    lib = _lib.load()
    v = _view(8, 300, 0.1)
    ref = ctypes.byref(v)
    T = lambda *a: _lib.StripView(8, 8, 8, *a)
    ok = T(0, 0, 48, 32, 1, 2)
    words = (ctypes.c_int64 * 3)()
    assert lib.slk_strip_words(ref, ctypes.byref(ok), words) == _lib.SLK_OK
    assert words[1] == 2 * 4 * 8 and words[2] == 7 * 2 + 7
    for bad, text in ((T(0, 0, 40, 32, 1, 1), "multiples of 16"), (T(0, 0, 272, 32, 1, 1), "256"),
                      (T(0, 0, 160, 32, 1, 2), "144"), (T(0, 0, 48, 0, 1, 1), "strip size"),
                      (T(8, 0, 48, 32, 1, 1), "no rows"), (T(1, 1, 48, 32, 1, 1), "row order")):
        assert lib.slk_strip_words(ref, ctypes.byref(bad), words) == _lib.SLK_EINVAL
        assert text in lib.slk_last_error().decode()
    need = lib.slk_strip_layout_bytes(300, 65)
    assert need == 4 * 300 * 128
    call = lambda t, N, ws, n: lib.slk_sddmm_strips(ref, ctypes.byref(t), 16, 16, N, 16, None, ws, n,
                                                    None)
    assert call(ok, 0, 16, need) == _lib.SLK_EINVAL and "N outside" in lib.slk_last_error().decode()
    assert call(ok, 65, 16, need - 1) == _lib.SLK_EINVAL
    assert "workspace" in lib.slk_last_error().decode()
    assert call(ok, 65, 8, need) == _lib.SLK_EINVAL


def test_more_rows_than_the_build_can_take_stay_with_slk_sddmm():
    M = 4 * 256 * 65535
    v = lambda m: _lib.CsrView(m, 64, 20 * m, 8, 8, 8, 8, 8)
    words = (ctypes.c_int64 * 3)()
    T = _lib.StripView(8, 8, 8, 0, 0, 48, 32, 1, 2)
    assert _lib.load().slk_strip_words(ctypes.byref(v(M)), ctypes.byref(T), words) == _lib.SLK_OK
    assert _lib.load().slk_strip_words(ctypes.byref(v(M + 1)), ctypes.byref(T), words) == _lib.SLK_EINVAL
    assert _lib.strip_choose(v(1 << 20), 1001)[0] is not None
    assert _lib.strip_choose(v(M + 1), 1001)[0] is None
