"""A PrefillPlan used on another stream than the one that built it: that
stream waits for the plan's transfer and the allocator learns of the use, on
the CPU with recorded stand-ins for the streams."""

import pytest
import torch

import naivllm_amd.layers.attention as at


class Stream:
    def __init__(self, name):
        self.cuda_stream, self.waits = name, []

    def wait_event(self, event):
        self.waits.append(event)


class Event:
    def __init__(self):
        self.on = None

    def record(self, stream):
        self.on = stream


class Work:
    def __init__(self):
        self.uses = []

    def record_stream(self, stream):
        self.uses.append(stream)


@pytest.fixture
def streams(monkeypatch):
    built, capturing = Stream("built"), [False]
    monkeypatch.setattr(torch.cuda, "get_device_properties", lambda d: type("P", (), {"multi_processor_count": 256}))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing[0])
    monkeypatch.setattr(torch.cuda, "current_stream", lambda d=None: built)
    monkeypatch.setattr(torch.cuda, "Event", Event)
    real = at._prefill_work
    monkeypatch.setattr(at, "_prefill_work", lambda *a: real(*a[:-1], False))
    return built, capturing


def make():
    plan = at.PrefillPlan([40], [40], 2, 1, 16, torch.device("cpu"))
    plan.work = Work()
    return plan


def test_the_building_stream_needs_no_wait(streams):
    plan = make()
    assert plan.ready.on is streams[0]
    plan.use_on(streams[0])
    assert streams[0].waits == [] and plan.work.uses == []


def test_another_stream_waits_and_is_recorded(streams):
    plan, other = make(), Stream("other")
    plan.use_on(other)
    assert other.waits == [plan.ready] and plan.work.uses == [other]


def test_a_capture_holds_no_outside_event(streams):
    plan, other = make(), Stream("other")
    streams[1][0] = True
    plan.use_on(other)
    assert other.waits == [] and plan.work.uses == []


def test_rows_of_a_step_of_few_and_their_streams(streams, monkeypatch):
    real = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, pin_memory=False, **k: real(*a, **k))
    rows, other = at.PrefillRows([3, 1, 2], [10, 1, 2], torch.device("cpu")), Stream("other")
    assert rows.context_lens.tolist() == [10, 1, 2] and rows.positions.tolist() == [7, 8, 9, 0, 0, 1]
    assert rows.cu_seqlens_q.tolist() == [0, 3, 4, 6] and rows.cu_seqlens_q.dtype == torch.int32 and rows.max_q_len == 3
    rows.work = Work()
    rows.use_on(other)
    assert other.waits == [rows.ready] and rows.work.uses == [other]


@pytest.mark.parametrize("ql,kl", [([0], [4]), ([5], [4]), ([1, 1], [4])])
def test_rows_of_bad_lengths_are_refused(streams, ql, kl):
    with pytest.raises(ValueError):
        at.PrefillRows(ql, kl, torch.device("cpu"))


def test_views_at_odd_offsets_are_copied():
    base = torch.arange(4 * 2 * 64 + 8, dtype=torch.bfloat16)
    for off in (0, 8):  # whole 16 bytes
        t = base[off:off + 512].view(4, 2, 64)
        assert at._aligned(t) is t
    for off in (1, 4):
        t = base[off:off + 512].view(4, 2, 64)
        assert t.is_contiguous() and at._aligned(t).data_ptr() % 16 == 0 and torch.equal(at._aligned(t), t)
