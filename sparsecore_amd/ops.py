"""sparsecore_amd.ops — spmm, its autograd Function and the transpose cache.

Drop-in for ``sparselab/ops.py``: same public ``spmm(W, X, *, kernel)``, same
``_SpMMFunction.apply(W_values, W, X, kernel)`` contract, same
``_transpose_cache`` / ``_cached_transpose`` / ``_clear_transpose_cache``
(cache entries are ``(topology_version, (nrows, ncols), WT, perm)``).

Every kernel runs on the HIP device through the C-ABI library:

    forward  Y  = W·X               slk_spmm                 (ops.py:144-165)
    backward dW = SDDMM(dY, X)      slk_sddmm                (ops.py:186-192)
             WT = cached transpose  slk_transpose_refresh on a hit,
                                    slk_transpose_count/fill on a miss (ops.py:70-99)
             dX = WT·dY             slk_spmm on WT           (ops.py:201-203)

Tensors on the CPU are rejected with RuntimeError (the reference rejected
non-CPU tensors the same way; this build is GPU-only and has no CPU path).
"""

from __future__ import annotations

import weakref

import torch

from . import _lib, layout
from .layout import PaddedCSR, transpose_with_perm, transposes_with_perm

__all__ = ["spmm", "dense_grad"]

_KERNELS = ("auto", "simd", "scalar")

# Key: id(W). Value: (topology_version, (nrows, ncols), WT, perm).
_transpose_cache: dict[int, tuple[int, tuple[int, int], PaddedCSR, torch.Tensor]] = {}


def _drop_entry(key: int) -> None:
    _transpose_cache.pop(key, None)


def _cached_transpose(W: PaddedCSR) -> PaddedCSR:
    """W's transpose, rebuilt only when W's topology changes (ops.py:70-99).

    Hit (same id, topology_version and shape): refresh the live WT values from
    W.values through perm on the device and return the same WT object.
    Miss: rebuild on the device and store the entry. Entries are dropped when
    W is garbage collected, so a recycled id() can never return a stale WT.
    """
    WT, perm, fresh = _transpose_entry(W)
    if not fresh:
        _lib.transpose_refresh(W.values, perm, WT.values)
    return WT


def _transpose_entry(W: PaddedCSR):
    """(WT, perm, fresh) from the transpose cache, rebuilt when W's topology
    changed; fresh: rebuilt by this call, with W's values."""
    key = id(W)
    cur_version = W.topology_version
    cur_shape = (int(W.nrows), int(W.ncols))
    cached = _transpose_cache.get(key)
    if cached is not None and cached[0] == cur_version and cached[1] == cur_shape:
        if torch.cuda.is_current_stream_capturing():
            W._pin(cached)  # the graph reads WT's arrays and perm
        return cached[2], cached[3], False
    WT, perm = transpose_with_perm(W)
    if cached is None:
        weakref.finalize(W, _drop_entry, key)
    _transpose_cache[key] = (cur_version, cur_shape, WT, perm)
    return WT, perm, True


def _rigl_update_cached(W: PaddedCSR, k_drop: int, dY: torch.Tensor, X: torch.Tensor) -> None:
    """``W._rigl_update(k_drop, dY, X)``, then W's cached transpose rebuilt for
    the new topology, as ``_cached_transpose`` would on its next call, with one
    host read for both: the rebuild is queued right behind the row rewrite,
    its slot arrays sized from the live slots before the update (rows only
    shrink), and its capacity read with the RigL counts. Without a cached
    transpose of W this is ``W._rigl_update``."""
    key = id(W)
    if key not in _transpose_cache:
        W._rigl_update(k_drop, dY, X)
        return
    staged = {}

    def then():
        staged["t"] = layout._transpose_queue(W, 0.2, W.nnz)
        return staged["t"]["counts"], finish

    def finish(host):
        if host is None:  # the exact path rewrote W after the queued rebuild
            _cached_transpose(W)
            return
        WT, perm = layout._transpose_take(W, staged["t"], host, W.nnz)
        _transpose_cache[key] = (W.topology_version, (int(W.nrows), int(W.ncols)), WT, perm)

    W._rigl_update(k_drop, dY, X, then=then)


def _cached_transpose_structure(W: PaddedCSR):
    """(WT, perm) from the transpose cache, rebuilt when W's topology changed
    (as ``_cached_transpose``) but without refreshing WT's values: for a
    caller that reads W's values through perm (slk_backward_fused). The next
    ``_cached_transpose`` refreshes them as on every hit."""
    return _transpose_entry(W)[:2]


def _rebuild_stale_transposes(Ws) -> None:
    """Rebuilds, in one batch (one device->host read for all), the cached
    transposes of those matrices whose entry exists but whose topology has
    changed — what the next backward of each would otherwise rebuild one by
    one, each with its own host read. Called by SET / RigL after a rewrite."""
    stale = []
    for W in Ws:
        cached = _transpose_cache.get(id(W))
        if cached is not None and (cached[0] != W.topology_version or
                                   cached[1] != (int(W.nrows), int(W.ncols))):
            stale.append(W)
    for W, (WT, perm) in zip(stale, transposes_with_perm(stale)):
        _transpose_cache[id(W)] = (W.topology_version, (int(W.nrows), int(W.ncols)), WT, perm)


def _clear_transpose_cache() -> None:
    """Testing utility: clear all cache entries. Not part of the public API."""
    _transpose_cache.clear()


# Phased gather sweep for slk_spmm (slk_csr.phase_lo) where X is far beyond
# the L2s: phases of at most _PHASE_X_ROWS X rows, so that the 1 KB pieces of
# one 256-column tile that a phase gathers (4 MiB) stay in an XCD's L2
# (measured on 16384^2 at 99%: forward 4.10 -> 2.49 ms with 4 phases, 2.90
# with 8, 4.16 with 16). Not for a matrix whose columns are skewed (the
# transpose of one with heavy rows): most of its gathers hit a few hot X rows
# that stay cached anyway, and phases only add passes (the same layer's dX
# 1.75 -> 2.08 ms). slk_spmm uses the bounds only on its 16-byte gather path;
# its LDS-staged kernel, which streams X once per workgroup, ignores them.
_PHASE_MIN_X_BYTES = 128 << 20
_PHASE_X_ROWS = 4096


# Binned slot stream for slk_spmm's LDS-staged kernel (slk_csr.bin_*). Row quads,
# which are asked first, take nearly every shape that passes these bars (all but
# 142 of 48987 sampled); what reaches it is the rest of them, captured calls whose
# quads no warm-up kept, and calls that found no memory for quads. For
# matrices without heavy rows where N is large, each staged X element is
# expected to serve at least _BIN_MIN_REUSE rows of a workgroup (density x
# rows per workgroup; fewer, and gathering X rows directly is faster), and a
# wave's rows are expected to hold at most _BIN_MAX_PER_CHUNK slots per
# staged chunk (its window holds 64; a chunk with more takes extra passes).
# Rows per wave and halves are the first of _BIN_SHAPES that qualifies (more
# rows per workgroup stage each X chunk for more rows; two halves halve the
# per-slot overhead per fma). Measured on 16384^2 x 4096 (same bits): the
# 95% layer's input gradient 5.80 -> 5.53 ms at 8 x 2; its forward, whose
# heavy rows run beside the light ones, 6.0 ms on the two-stream path against
# 6.43 binned; at 99% the gather kernel (1.79 ms) beats any binned shape
# (3.5 ms and up: staging all of X per workgroup dominates). Only from
# _BIN_MIN_NNZ live slots: on the 10M- and 60M-GPT layers (0.1-0.5 M slots)
# the binned kernel runs no faster than the LDS kernel, while its build (one
# per topology version; SET rewrites every layer every step) and its view
# cost step time: 60M-GPT + SET 43.0 -> 46.4 ms/step, 10M-GPT 11.1 -> 11.7.
_BIN_MIN_NNZ = 4_000_000
_BIN_MIN_N = 1024
_BIN_MIN_REUSE = 4.0
_BIN_MAX_PER_CHUNK = 48
_BIN_MIN_BLOCKS = 192
_BIN_SHAPES = ((8, 2), (4, 2), (2, 2), (8, 1), (4, 1), (1, 2))


def _bin_shape(W: PaddedCSR, K: int, N: int):
    """(rows per wave, halves) of the binned stream slk_spmm should get for W
    and an N-column X, or None."""
    if N < _BIN_MIN_N or N % 4 or K == 0 or W.nnz < _BIN_MIN_NNZ:
        return None
    first, slots = W._bin_coverage()
    rows = W.nrows - first
    if first > 0 or rows <= 0 or slots <= 0:
        return None
    density = slots / (rows * K)
    for rw, h in _BIN_SHAPES:
        kc = 80 // h
        if -(-K // kc) > _lib.BIN_MAX_CHUNKS:
            continue
        if rw * kc * density > _BIN_MAX_PER_CHUNK or density * 16 * rw < _BIN_MIN_REUSE:
            continue
        if -(-rows // (16 * rw)) * -(-N // (256 * h)) < _BIN_MIN_BLOCKS:
            continue
        return rw, h
    return None


# Schedule overrides for tests and measurement (the launchers' own choices
# otherwise; results keep their bits either way): "spmm_phases" = n forces
# n column phases on slk_spmm's gather path (<= 1: none); "seg" = (block
# columns, slots per segment) forces that segment list on slk_sddmm, () none;
# "bin_shape" = (rows per wave, halves) forces that binned stream on
# slk_spmm, False none; "quad" = 1 or 2 forces row quads of that many halves,
# 0 none; "strips" = (block, slots, per_wave, parts) forces those strips for dW,
# None none.
_overrides: dict[str, object] = {}


# Row quads (slk_spmm_quad) instead of slk_spmm where slk_quad_halves expects
# them to be faster: layers of some 5% density and up at N of about 1000 and up,
# all but the smallest where N is not a multiple of 4 (2304 x 768, N = 8192,
# 20%: 238 -> 190 us; 3072 x 768, N = 1001, 10%: 87 -> 37; 4096^2 x 4096, 10%:
# 566 -> 462). Below _QUAD_MIN_WORK live slots x N no shape gains (the smallest
# that does, 1152 x 384 at 10% and N = 1001, has 4.4e7), so the call is spared.
_QUAD_MIN_WORK = 30_000_000

# Under graph capture a call whose plain kernel reads nothing but the matrix's own
# arrays records the build of its quads or strips with itself, so that a replay
# follows the rows as they are, as the plain kernel's would, and the graph owns all
# that it reads. The build adds 9-20 us to each replay (4096 x 1024 to 4096^2 at
# 30% the most), which they repay from this many live slots x N on: where N is
# not a multiple of 4 (1152 x 384 at 30%, N = 1001: forward 49 -> 44 us, dW 42 ->
# 40; 2304 x 768 at 30%, N = 1001: 161 -> 74, 145 -> 65; 4096 x 1024 at 10%, N =
# 333, below the line: dW 53 -> 57) and where it is (2304 x 768 at 30%, N = 8192:
# forward 289 -> 269; 3072 x 768 at 30%, N = 2048, below: 107 -> 109). Where the
# plain kernel needs a schedule of the topology itself, as the segment kernel does,
# a captured call runs on the quads or strips that its warm-up kept.
_CAPTURED_MIN_WORK = 150_000_000
_CAPTURED_MIN_WORK_ALIGNED = 3_000_000_000


def _recording_pays(W: PaddedCSR, N: int) -> bool:
    """Whether a captured call gains by quads or strips that every replay builds."""
    return W.nnz * N >= (_CAPTURED_MIN_WORK if N % 4 else _CAPTURED_MIN_WORK_ALIGNED)


# The estimates behind quads and strips take rows of like length, and refuse
# heavy rows, which only views from _ORDER_MIN_ROWS rows on count. Below that,
# where more than one row in 32 is heavy (Zipf(0.5) and Zipf(1.1) row lengths,
# 256 to 2000 rows, 784 to 4096 columns, 3% to 25%; each against slk_spmm or
# slk_sddmm): at N a multiple of 4 quads are faster up to 512 rows (1.0-1.7x) and
# at 3% (1.0-2.3x) but slower above (0.73-1.1x, most at 1024 x 2048, 10%: 271 ->
# 370 us); at other N they are always faster (1.1-3.5x). Strips are slower at N a
# multiple of 4 (0.45-1.06x: 2000 x 4096 at 3%, N = 2048: 94 -> 207 us), faster at
# other N (1.06-4.7x), except below some 4e8 slots x N (2000 x 784 at 10%, N =
# 1001: 52 -> 79).
_SKEW_QUAD_MAX_ROWS = 512
_SKEW_QUAD_MAX_DENSITY = 1 / 16
_SKEW_STRIP_MIN_WORK = 400_000_000


def _skewed(W: PaddedCSR) -> bool:
    return W.nrows < W._ORDER_MIN_ROWS and W._skewed()


def _skew_slows_quads(W: PaddedCSR, N: int) -> bool:
    return N % 4 == 0 and W.nrows > _SKEW_QUAD_MAX_ROWS and \
        W.nnz >= _SKEW_QUAD_MAX_DENSITY * W.nrows * W.ncols and _skewed(W)


def _skew_slows_strips(W: PaddedCSR, N: int) -> bool:
    return (N % 4 == 0 or W.nnz * N < _SKEW_STRIP_MIN_WORK) and _skewed(W)


# What quads and strips are taken for is kept with W's view, by N (dW: (N,)): it
# depends on shape, capacity, live slots and the counts of heavy and dense rows,
# which last as long as the view's row counts. Not while a kernel-choice knob is
# forced, and not from a captured call, where the rows' skew may be unknown.
_ROUTES = 64


def _keep_route(routes: dict, key, choice):
    if not _lib.FORCED_KNOBS and not torch.cuda.is_current_stream_capturing():
        if len(routes) >= _ROUTES:
            routes.clear()
        routes[key] = choice
    return choice


def _quad_plan(W: PaddedCSR, K: int, N: int, mapped: bool = False):
    """(halves, capturing, recorded) of the row quads to run W on a K x N X with;
    None: slk_spmm. mapped: W is a cached transpose, run through its slot map."""
    if _overrides:
        halves = _overrides.get("quad")
        if halves is not None:
            capturing = torch.cuda.is_current_stream_capturing()
            return (int(halves), capturing, not mapped) if halves else None
        if "bin_shape" in _overrides or "spmm_phases" in _overrides:
            return None
    if W.nnz * N < _QUAD_MIN_WORK:
        return None
    view = W._view()
    halves = view.routes.get(N)
    if halves is None or _lib.FORCED_KNOBS:
        halves = _lib.quad_halves(view, N)
        if halves and _skew_slows_quads(W, N):
            halves = 0
        _keep_route(view.routes, N, halves)
    if not halves:
        return None
    if not torch.cuda.is_current_stream_capturing():
        return halves, False, False
    if mapped or _spmm_scheduled(W, K, N):
        return (halves, True, False) if W._has("_quads_kept", (halves, mapped)) else None
    # (a graph cannot read the exact size of large quads, and would hold the bound)
    if not _recording_pays(W, N) or _lib.quad_bytes(view, halves) > _lib.QUAD_READ_BYTES:
        return None
    return halves, True, True


def _quad_halves(W: PaddedCSR, K: int, N: int, mapped: bool = False) -> int:
    """64-column halves (1 or 2) of _quad_plan's quads; 0: slk_spmm."""
    plan = _quad_plan(W, K, N, mapped)
    return plan[0] if plan else 0


def _spmm_quads(W: PaddedCSR, values: torch.Tensor, X: torch.Tensor, Y: torch.Tensor, plan,
                perm: torch.Tensor | None = None, bias: torch.Tensor | None = None) -> bool:
    """Y = W·X (+ bias) through W's row quads. False, with nothing launched and
    W's quads given up, where the memory for them is not to be had: slk_spmm needs
    none."""
    halves, capturing, recorded = plan
    try:
        _lib.spmm_quad(W._view(), W._quads(halves, perm, capturing, recorded), values, X, Y, bias)
    except torch.OutOfMemoryError:
        W._quads_kept = (-1, {})
        return False
    return True


def _phases(W: PaddedCSR, K: int, N: int) -> int:
    """Column phases of slk_spmm's gather path where X is far beyond the L2s and
    W's columns are not skewed; 0: one sweep."""
    if 4 * K * N >= _PHASE_MIN_X_BYTES and K > _PHASE_X_ROWS and not W._cols_skewed:
        return -(-K // _PHASE_X_ROWS)
    return 0


def _spmm_scheduled(W: PaddedCSR, K: int, N: int) -> bool:
    """Whether slk_spmm would run W by a schedule of its topology."""
    return _phases(W, K, N) > 0 or _bin_shape(W, K, N) is not None


def _spmm_view(W: PaddedCSR, X: torch.Tensor):
    """W's view for slk_spmm: with a binned slot stream where it pays (see
    above), else with phase bounds."""
    K, N = X.shape
    binned = _overrides.get("bin_shape")
    if binned is None:
        binned = _bin_shape(W, K, N)
    if binned:
        return W._view_binned(*binned)
    forced = _overrides.get("spmm_phases")
    phases = _phases(W, K, N) if forced is None else int(forced)
    return W._view_phased(phases) if phases > 1 else W._view()


def _launch_spmm(W: PaddedCSR, X: torch.Tensor, bias: torch.Tensor | None = None,
                 quads: bool = True) -> torch.Tensor:
    """W·X (+ bias per row); quads: not known to be out of the question."""
    Y = torch.empty((W.nrows, X.shape[1]), dtype=torch.float32, device=X.device)
    plan = _quad_plan(W, *X.shape) if quads else None
    if plan is None or not _spmm_quads(W, W.values, X, Y, plan, bias=bias):
        _lib.spmm(_spmm_view(W, X), X, Y, bias)
    return Y


# Segment schedule for dW (slk_csr.seg_start): from this many live slots at
# N >= 1024 (measured per layer: 1.4-1.8x on the 60M-GPT layers, 1.35x on the
# 10M-GPT QKV layer, 1.5x / 1.45x on the 16384^2 layer at 95% / 99%; the
# windowed kernel stays ahead on the 10M-GPT layers of 44-59 k slots).
_SEG_MIN_NNZ = 100_000
# X at least this large (far beyond the 4 MB L2 of an XCD) takes 128-column
# segment blocks where rows are dense enough.
_SEG_WIDE_MIN_X_BYTES = 128 << 20


def _seg_shape(W: PaddedCSR, K: int, N: int) -> tuple[int, int]:
    """(block columns, slots per segment) of the segment list: 128-column
    blocks of 8-slot segments where X is far beyond the L2s (each dY row is
    then fetched once per 128 columns instead of 64; waves skip the slots
    their segments lack, so short runs cost little: 16384^2 at 95% 5.65 ms
    against 6.53 for 64x8, at 99% 1.92 against 2.21 for 64x4); else 64
    columns, with 8 slots per segment where a row holds at least 4 live slots
    per block on average, else 4."""
    if 4 * K * N >= _SEG_WIDE_MIN_X_BYTES:
        return 128, 8
    density = W.nnz / max(1, W.nrows * W.ncols)
    return 64, 8 if density * 64 >= 4 else 4


# Dense rows (slk_csr.n_dense_rows) of a segmented dW run on the matrix cores
# where N is a multiple of 64 (the dense kernel's staged columns) and there
# are at least _DENSE_DW_MIN_ROWS of them: the segment kernel's time follows
# its (row, column block) pairs more than its slots, so a few dense rows
# taken out save little (16384^2 Zipf(1.1) x 4096: 95%, 622 dense rows,
# 5.47 -> 5.22 ms; 99%, 102 rows, 1.86 -> 2.04 ms). "dense_dw" = False in
# _overrides keeps them in the segment list, True takes any count.
_DENSE_DW_N = 64
_DENSE_DW_MIN_ROWS = 256


def _sddmm_view(W: PaddedCSR, X: torch.Tensor):
    """W's view for slk_sddmm: with a segment list where it pays (see above),
    without W's dense rows where the dense kernel takes them."""
    K, N = X.shape
    want = _overrides.get("dense_dw")
    skip = N % _DENSE_DW_N == 0 and N >= _DENSE_DW_N and want is not False and (
        want is True or W._view().n_dense_rows >= _DENSE_DW_MIN_ROWS)
    forced = _overrides.get("seg")
    if forced is not None:
        return W._view_segmented(*forced, skip_dense=skip) if forced else W._view()
    if _sddmm_scheduled(W, N):
        return W._view_segmented(*_seg_shape(W, K, N), skip_dense=skip)
    return W._view()


def _sddmm_scheduled(W: PaddedCSR, N: int) -> bool:
    """Whether slk_sddmm would run W by a segment list."""
    return W.nnz >= _SEG_MIN_NNZ and N >= 1024 and N % 4 == 0


# Strips (slk_sddmm_strips) instead of slk_sddmm where slk_strip_choose expects
# them to be faster: N not a multiple of 4 (1537 x 1000 at 20%, N = 1777: 194 ->
# 52 us), N below 1024 or too few slots for the segment list (512 x 784 at 20%, N
# = 8192: 159 -> 108), and layers around 3-5% and 20-40% (4096^2 x 4096 at 5%: 579
# -> 405; 2304 x 768 at 30%, N = 8192: 365 -> 283). Below _STRIP_MIN_WORK live
# slots x N no shape gains.
_STRIP_MIN_WORK = 30_000_000


def _strip_plan(W: PaddedCSR, N: int):
    """((block, slots, per_wave, parts), capturing, recorded) of the strips to run
    W's dW with at N columns; None: slk_sddmm."""
    if _overrides:
        if "strips" in _overrides:
            sizes = _overrides["strips"]
            return (sizes, torch.cuda.is_current_stream_capturing(), True) if sizes else None
        if "seg" in _overrides or "dense_dw" in _overrides:
            return None
    if W.nnz * N < _STRIP_MIN_WORK or \
            not _lib.FORCED_KNOBS.isdisjoint(("sddmm_g", "seg_lean", "seg_group")):
        return None
    view = W._view()
    sizes = view.routes.get((N,))
    if sizes is None:
        sizes = _lib.strip_choose(view, N)[0] or ()
        if sizes and _skew_slows_strips(W, N):
            sizes = ()
        _keep_route(view.routes, (N,), sizes)
    if not sizes:
        return None
    if not torch.cuda.is_current_stream_capturing():
        return sizes, False, False
    if _sddmm_scheduled(W, N):
        return (sizes, True, False) if W._has("_strips_kept", sizes) else None
    return (sizes, True, True) if _recording_pays(W, N) else None


def _strip_sizes(W: PaddedCSR, N: int):
    """_strip_plan's (block, slots, per_wave, parts); None: slk_sddmm."""
    plan = _strip_plan(W, N)
    return plan[0] if plan else None


def _launch_sddmm(W: PaddedCSR, dY: torch.Tensor, X: torch.Tensor, kernel: str,
                  dbias: torch.Tensor | None = None) -> torch.Tensor:
    dW = torch.empty(W.total_capacity, dtype=torch.float32, device=X.device)
    if kernel == "scalar":
        _lib.sddmm(W._view(), dY, X, dW, _lib.SLK_DW_SCALAR, dbias)
        return dW
    plan = _strip_plan(W, X.shape[1])
    if plan is not None:
        try:
            _lib.sddmm_strips(W._view(), W._strips(*plan), dY, X, dW, dbias)
            return dW
        except torch.OutOfMemoryError:  # for the strips or their copy of X
            W._strips_kept = (-1, {})
    _lib.sddmm(_sddmm_view(W, X), dY, X, dW, _lib.SLK_DW_SIMD, dbias)
    return dW


def _device_f32(t: torch.Tensor) -> torch.Tensor:
    return t.to(dtype=torch.float32).contiguous()


def _check_same_device(W: PaddedCSR, t: torch.Tensor, who: str, name: str) -> None:
    if t.device.type != "cuda":
        raise RuntimeError(
            f"{who}: {name} must be on a HIP (ROCm) device (got device={t.device}). "
            f"sparsecore_amd runs the padded-CSR kernels on the GPU only.")
    W._require_device(who)
    if W.device != t.device:
        raise RuntimeError(f"{who}: W is on {W.device} but {name} is on {t.device}")


class _SpMMFunction(torch.autograd.Function):
    """Autograd bridge for Y = W @ X with W a PaddedCSR (ops.py:127-210).

    The first input, ``W_values``, is the tensor autograd tracks (aliased with
    ``W.values`` by SparseLinear); the kernels read the weights through W, as
    the reference does. Backward returns dW aligned with W.values (length
    total_capacity, padding exactly 0) and dX = Wᵀ·dY. A gradient nobody asked
    for (``needs_input_grad`` False) is not computed.
    """

    @staticmethod
    def forward(ctx, W_values, W, X, kernel):
        ctx.save_for_backward(W_values, X)
        ctx.W = W
        ctx.kernel = kernel
        if kernel not in _KERNELS:
            raise ValueError(f"spmm: unknown kernel={kernel!r}. Expected one of: "
                             f"{sorted(_KERNELS)}.")
        _check_same_device(W, X, "spmm", "X")
        return _launch_spmm(W, _device_f32(X))

    @staticmethod
    def backward(ctx, dY):
        W_values, X = ctx.saved_tensors
        dW_values, dX = _spmm_backward(ctx.W, X, _as_row_major(dY), ctx.kernel,
                                       ctx.needs_input_grad[0], ctx.needs_input_grad[2])
        return dW_values, None, dX, None


# Small layers: the backward as one launch (slk_backward_fused) where dW,
# the transpose refresh and dX would each be a few microseconds of launch
# latency (a 512 x 784 layer at N = 256: 6.8 + 2.3 + 8.2 us in a graph): up
# to this many waves in the fused grid, one round of waves on the chip.
_FUSED_MAX_WAVES = 8192


def _fused_backward(W: PaddedCSR, N: int, kernel: str) -> bool:
    forced = _overrides.get("fused_backward")
    if forced is not None:
        return bool(forced) and kernel != "scalar"
    if kernel == "scalar" or N == 0:
        return False
    waves = W.ncols * -(-N // 64) + -(-W.total_capacity // 16)
    return waves <= _FUSED_MAX_WAVES


def _spmm_backward(W: PaddedCSR, X: torch.Tensor, dY_f32: torch.Tensor, kernel: str,
                   need_dw: bool, need_dx: bool, dbias: torch.Tensor | None = None):
    """dW on the live slots (SDDMM) and dX = Wᵀ·dY through the transpose cache
    (ops.py:167-210); a gradient that is not needed is not computed. With
    ``dbias`` (and dW needed) the dW launch also writes dY's row sums there.
    Small layers run both in one launch, W's values read through the
    transpose's slot map instead of a refresh (same bits)."""
    if need_dw and need_dx and _fused_backward(W, dY_f32.shape[1], kernel):
        WT, perm = _cached_transpose_structure(W)
        X32 = _device_f32(X)
        dW_values = torch.empty(W.total_capacity, dtype=torch.float32, device=X32.device)
        dX = torch.empty(W.ncols, dY_f32.shape[1], dtype=torch.float32, device=X32.device)
        _lib.backward_fused(W._view(), WT._view(), perm, dY_f32, X32, dW_values, dbias, dX)
        return dW_values, dX
    dW_values = dX = None
    if need_dw:
        dW_values = _launch_sddmm(W, dY_f32, _device_f32(X), kernel, dbias)
    if need_dx:
        WT, perm, fresh = _transpose_entry(W)
        plan = _quad_plan(WT, *dY_f32.shape, mapped=True)
        if plan is not None:  # through W's values: no refresh of WT's
            dX = torch.empty((W.ncols, dY_f32.shape[1]), dtype=torch.float32, device=W.device)
            if not _spmm_quads(WT, W.values, dY_f32, dX, plan, perm):
                dX = None
        if dX is None:
            if not fresh:
                _lib.transpose_refresh(W.values, perm, WT.values)
            dX = _launch_spmm(WT, dY_f32, quads=False)
    return dW_values, dX


def _as_row_major(t: torch.Tensor) -> torch.Tensor:
    """``t.to(float32).contiguous()`` where a transposed view is copied by the
    library's tiled transpose (slk_transpose_dense) instead of torch's
    strided copy: the `dY.contiguous()` of ops.py:174, bit for bit."""
    t = t.to(dtype=torch.float32)
    if t.is_contiguous():
        return t
    if t.dim() == 2 and t.t().is_contiguous() and t.device.type == "cuda":
        out = torch.empty(t.shape, dtype=torch.float32, device=t.device)
        _lib.transpose_dense(t.t(), out)
        return out
    return t.contiguous()


def _narrow_layer(W: PaddedCSR) -> bool:
    """A layer small enough for the narrow path (slk_spmm_t forward,
    slk_backward_narrow backward): at most 64 output rows and 8192 slots."""
    return W.nrows <= _lib.NARROW_MAX_ROWS and W.total_capacity <= _lib.NARROW_MAX_CAPACITY


class _SparseLinearFunction(torch.autograd.Function):
    """SparseLinear's ``Y = W @ x_flatᵀ (+ bias[:, None])`` as one autograd node
    (sparselab/nn.py:229-241 with ops.py:127-210 inside).

    Takes the token-major input x_flat (N x K). Returns Y feature-major
    (M x N), whose ``.t()`` is the layer output, or — for a narrow layer
    (``_narrow_layer``) — the layer output itself, token-major (N x M)
    contiguous. The layout changes of the reference (``x_flat.t().contiguous()``,
    the bias add, ``dY.contiguous()``) are done by the library: the transpose
    by slk_transpose_dense — free when x_flat is the transposed view a
    previous SparseLinear returned — and the bias add inside the SpMM store
    (slk_spmm_bias / slk_spmm_t: the bits of the separate float32 add).
    Backward is ``_SpMMFunction``'s, plus dbias = Σ_n dY[:, n] computed in the
    dW launch (slk_sddmm_bias); a narrow layer does all three gradients in one
    launch from the token-major gradient (slk_backward_narrow), with no
    transpose cache. dx is returned as the transposed view of dX (K x N).
    """

    @staticmethod
    def forward(ctx, W_values, bias, W, x_flat, kernel):
        if kernel not in _KERNELS:
            raise ValueError(f"spmm: unknown kernel={kernel!r}. Expected one of: "
                             f"{sorted(_KERNELS)}.")
        _check_same_device(W, x_flat, "spmm", "X")
        X = _as_row_major(x_flat.t())
        if bias is not None:
            _check_same_device(W, bias, "spmm", "bias")
            if bias.dtype != torch.float32 or bias.shape != (W.nrows,):
                raise ValueError(f"spmm: bias must be float32 of shape ({W.nrows},), got "
                                 f"{bias.dtype} {tuple(bias.shape)}")
            bias = bias.contiguous()
        ctx.save_for_backward(W_values, X)
        ctx.W = W
        ctx.kernel = kernel
        ctx.narrow = _narrow_layer(W)
        if ctx.narrow:
            Yt = torch.empty(X.shape[1], W.nrows, dtype=torch.float32, device=X.device)
            _lib.spmm_t(W._view(), X, Yt, bias)
            return Yt
        return _launch_spmm(W, X, bias)

    @staticmethod
    def backward(ctx, dY):
        W_values, X = ctx.saved_tensors
        if ctx.narrow:
            return _narrow_backward(ctx, X, dY)
        dY_f32 = _as_row_major(dY)
        need_dw, need_db = ctx.needs_input_grad[0], ctx.needs_input_grad[1]
        dbias = None
        if need_db:  # fused into the dW launch when dW is computed too
            dbias = torch.empty(dY_f32.shape[0], dtype=torch.float32, device=dY_f32.device)
            if not need_dw:
                torch.sum(dY_f32, dim=1, out=dbias)
        dW_values, dX = _spmm_backward(ctx.W, X, dY_f32, ctx.kernel, need_dw,
                                       ctx.needs_input_grad[3], dbias if need_dw else None)
        return dW_values, dbias, None, (dX.t() if dX is not None else None), None


def _narrow_backward(ctx, X: torch.Tensor, dYt: torch.Tensor):
    """Gradients of a narrow layer from the token-major output gradient."""
    W = ctx.W
    dev = X.device
    dYt = dYt.to(torch.float32).contiguous()
    need_dw, need_db, need_dx = (ctx.needs_input_grad[0], ctx.needs_input_grad[1],
                                 ctx.needs_input_grad[3])
    dW = torch.empty(W.total_capacity, dtype=torch.float32, device=dev) if need_dw else None
    dbias = torch.empty(W.nrows, dtype=torch.float32, device=dev) if need_db else None
    dX = torch.empty(X.shape, dtype=torch.float32, device=dev) if need_dx else None
    order = _lib.SLK_DW_SCALAR if ctx.kernel == "scalar" else _lib.SLK_DW_SIMD
    _lib.backward_narrow(W._view(), dYt, X, dW, dbias, dX, order)
    return dW, dbias, None, (dX.t() if dX is not None else None), None


def spmm(W: PaddedCSR, X: torch.Tensor, *, kernel: str = "auto") -> torch.Tensor:
    """Y = W @ X for a PaddedCSR W (M x K) and a dense 2-D X (K x N) on the GPU.

    Same contract as sparselab.ops.spmm (ops.py:217-331) except for the
    device: X (and W) must live on the HIP device. Any float dtype is
    converted to float32. If X requires grad the call goes through the
    autograd Function. ``kernel`` ("auto", "simd", "scalar") selects the dW
    summation order of the reference kernel of that name; the forward result
    is the same for all three.

    Raises TypeError (wrong W / X type), RuntimeError (tensor not on the HIP
    device) and ValueError (X not 2-D, shape mismatch, unknown kernel).
    """
    if not isinstance(W, PaddedCSR):
        raise TypeError(f"spmm: W must be a sparselab.PaddedCSR, got {type(W).__name__}")
    if not isinstance(X, torch.Tensor):
        raise TypeError(f"spmm: X must be a torch.Tensor, got {type(X).__name__}")
    if X.device.type != "cuda":
        raise RuntimeError(
            f"spmm: X must be on a HIP (ROCm) device (got device={X.device}). "
            f"sparsecore_amd runs the padded-CSR kernels on the GPU only.")
    if X.dim() != 2:
        raise ValueError(f"spmm: X must be 2-D, got shape={tuple(X.shape)}")
    if kernel not in _KERNELS:
        raise ValueError(f"spmm: unknown kernel={kernel!r}. Expected one of: "
                         f"{sorted(_KERNELS)}.")
    _check_same_device(W, X, "spmm", "X")
    X_f32 = _device_f32(X)
    W_values_t = W.values
    if X_f32.requires_grad or W_values_t.requires_grad:
        return _SpMMFunction.apply(W_values_t, W, X_f32, kernel)
    return _launch_spmm(W, X_f32)


def dense_grad(dY: torch.Tensor, X: torch.Tensor) -> torch.Tensor:
    """G = dY @ Xᵀ (M x K) for dense dY (M x N) and X (K x N) on the GPU.

    Mirrors ``_core.dense_grad`` (csrc/bindings.cpp:445-485): 2-D inputs,
    converted to contiguous float32, ValueError on a rank or inner-dimension
    mismatch with the reference's message. Every element is the reference
    build's running sum over N in order, so G is bit-identical to
    csrc/kernels/dense_grad.cpp:57-83.
    """
    for name, t in (("dY", dY), ("X", X)):
        if not isinstance(t, torch.Tensor):
            raise TypeError(f"dense_grad: {name} must be a torch.Tensor, got {type(t).__name__}")
        if t.dim() != 2:
            raise ValueError(f"dense_grad: {name} must be 2-D, got ndim={t.dim()}.")
        if t.device.type != "cuda":
            raise RuntimeError(f"dense_grad: {name} must be on a HIP (ROCm) device "
                               f"(got device={t.device}).")
    if dY.device != X.device:
        raise RuntimeError(f"dense_grad: dY is on {dY.device} but X is on {X.device}")
    M, N = dY.shape
    K, N_x = X.shape
    if N != N_x:
        raise ValueError(f"dense_grad: dY.shape[1]={N} must equal X.shape[1]={N_x} "
                         f"(shared inner dim N).")
    G = torch.empty((M, K), dtype=torch.float32, device=dY.device)
    _lib.dense_grad(_device_f32(dY), _device_f32(X), M, K, N, False, G)
    return G


def _dense_grad_token_major(dy: torch.Tensor, x: torch.Tensor) -> torch.Tensor:
    """G = dyᵀ @ x for token-major dy (N x M) and x (N x K): the same G as
    ``dense_grad(dy.t(), x.t())``, bit for bit, without the transpose copies."""
    N, M = dy.shape
    K = x.shape[1]
    G = torch.empty((M, K), dtype=torch.float32, device=dy.device)
    _lib.dense_grad(_device_f32(dy), _device_f32(x), M, K, N, True, G)
    return G
