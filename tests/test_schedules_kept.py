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


def _build(made):
    def build():
        a = _Array()
        made.append(a)
        return a, (a,)
    return build


def test_another_stream_waits_for_the_build_and_is_a_user_of_its_arrays(W, gpu):
    made = []
    first = W._kept("_quads_kept", 1, _build(made))
    assert W._kept("_quads_kept", 1, _build(made)) is first and gpu.log == []
    for stream in (2, 3, 2, 1):
        gpu.stream = stream
        assert W._kept("_quads_kept", 1, _build(made)) is first and len(made) == 1
    assert gpu.log == [("record", 1), ("wait", 2, "event of 1"),
                       ("record", 1), ("wait", 3, "event of 1")]
    assert first.users == [2, 3]


def test_every_key_of_a_topology_is_kept(W, gpu):
    """Nothing built for this topology is dropped while it lasts: a captured
    call may hold its address."""
    made = []
    got = [W._kept("_strips_kept", n, _build(made)) for n in range(8)]
    assert [W._kept("_strips_kept", n, _build(made)) for n in range(8)] == got and len(made) == 8
    W.rewrite_row(0, [1], [1.0])
    assert W._kept("_strips_kept", 0, _build(made)) is not got[0]


def test_a_capture_pins_what_it_reads_until_one_under_a_newer_topology(W, gpu):
    made = []
    old = W._kept("_segs_kept", 1, _build(made))
    gpu.capturing, gpu.stream = True, 2
    assert W._kept("_segs_kept", 1, _build(made)) is old
    assert W._kept("_segs_kept", 1, _build(made)) is old
    assert gpu.log == [], "no wait for an event of before the capture"
    assert [b.value for b in W._pinned[1]] == [old]
    gpu.capturing, gpu.stream = False, 1
    W.rewrite_row(0, [1], [1.0])
    new = W._kept("_segs_kept", 1, _build(made))
    assert new is not old and [b.value for b in W._pinned[1]] == [old]
    gpu.capturing = True
    W._kept("_segs_kept", 1, _build(made))
    assert [b.value for b in W._pinned[1]] == [new]


def test_what_a_capture_builds_is_the_graphs_alone(W, gpu):
    made = []
    gpu.capturing = True
    W._kept("_phases_kept", 1, _build(made))
    gpu.capturing = False
    W._kept("_phases_kept", 1, _build(made))
    assert len(made) == 2
    # recorded: anew under capture though a kept one is there, which stays
    kept = W._kept("_quads_kept", 1, _build(made), recorded=True)
    gpu.capturing = True
    assert W._kept("_quads_kept", 1, _build(made), recorded=True) is not kept
    gpu.capturing = False
    assert W._kept("_quads_kept", 1, _build(made), recorded=True) is kept and len(made) == 4
