"""How PaddedCSR keeps lazily built device state (row orders, schedules) between
calls, without a device: what a call on another stream, under graph capture and
after a topology change is given. Streams and events are recorded stand-ins."""

from __future__ import annotations

import pytest
import torch

from sparsecore_amd import layout


class _Array:
    """A device array as far as the keeping sees it."""

    device = torch.device("cuda", 0)

    def __init__(self):
        self.users = []

    def record_stream(self, stream):
        self.users.append(stream.cuda_stream)


class _Stream:
    def __init__(self, number, log):
        self.cuda_stream, self.log = number, log

    def record_event(self):
        self.log.append(("record", self.cuda_stream))
        return f"event of {self.cuda_stream}"

    def wait_event(self, event):
        self.log.append(("wait", self.cuda_stream, event))


@pytest.fixture
def gpu(monkeypatch):
    class State:
        stream, capturing, log = 1, False, []

    st = State()
    st.log = []
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: _Stream(st.stream, st.log))
    monkeypatch.setattr(torch.cuda, "ExternalStream", lambda raw, device=None: _Stream(raw, st.log))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: st.capturing)
    monkeypatch.setattr(layout, "_raw_stream", lambda index: st.stream)
    return st


@pytest.fixture
def W():
    return layout.from_dense(torch.eye(4))


def _get(W, gpu, made, name, key, recorded=False):
    """What the schedules of layout.PaddedCSR do: find, else build and keep."""
    a = W._find(name, key, gpu.capturing, recorded)
    if a is None:
        a = _Array()
        made.append(a)
        W._keep(name, key, a, (a,), gpu.capturing)
    return a


def test_another_stream_waits_for_the_build_and_is_a_user_of_its_arrays(W, gpu):
    made = []
    first = _get(W, gpu, made, "_quads_kept", 1)
    assert _get(W, gpu, made, "_quads_kept", 1) is first and gpu.log == []
    for stream in (2, 3, 2, 1):
        gpu.stream = stream
        assert _get(W, gpu, made, "_quads_kept", 1) is first and len(made) == 1
    assert gpu.log == [("record", 1), ("wait", 2, "event of 1"),
                       ("record", 1), ("wait", 3, "event of 1")]
    assert first.users == [2, 3]


def test_every_key_of_a_topology_is_kept(W, gpu):
    """Nothing built for this topology is dropped while it lasts: a captured
    call may hold its address."""
    made = []
    got = [_get(W, gpu, made, "_strips_kept", n) for n in range(8)]
    assert [_get(W, gpu, made, "_strips_kept", n) for n in range(8)] == got and len(made) == 8
    W.rewrite_row(0, [1], [1.0])
    assert _get(W, gpu, made, "_strips_kept", 0) is not got[0]


def test_a_capture_pins_what_it_reads_until_one_under_a_newer_topology(W, gpu):
    made = []
    old = _get(W, gpu, made, "_segs_kept", 1)
    gpu.capturing, gpu.stream = True, 2
    assert _get(W, gpu, made, "_segs_kept", 1) is old
    assert _get(W, gpu, made, "_segs_kept", 1) is old
    assert gpu.log == [], "no wait for an event of before the capture"
    assert [b.value for b in W._pinned[1]] == [old]
    gpu.capturing, gpu.stream = False, 1
    W.rewrite_row(0, [1], [1.0])
    new = _get(W, gpu, made, "_segs_kept", 1)
    assert new is not old and [b.value for b in W._pinned[1]] == [old]
    gpu.capturing = True
    _get(W, gpu, made, "_segs_kept", 1)
    assert [b.value for b in W._pinned[1]] == [new]


def test_what_a_capture_builds_is_the_graphs_alone(W, gpu):
    made = []
    gpu.capturing = True
    _get(W, gpu, made, "_phases_kept", 1)
    gpu.capturing = False
    _get(W, gpu, made, "_phases_kept", 1)
    assert len(made) == 2
    # recorded: anew under capture though a kept one is there, which stays
    kept = _get(W, gpu, made, "_quads_kept", 1, recorded=True)
    gpu.capturing = True
    assert _get(W, gpu, made, "_quads_kept", 1, recorded=True) is not kept
    gpu.capturing = False
    assert _get(W, gpu, made, "_quads_kept", 1, recorded=True) is kept and len(made) == 4
