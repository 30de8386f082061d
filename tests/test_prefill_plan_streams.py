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


def test_views_at_odd_offsets_are_copied():
    base = torch.arange(4 * 2 * 64 + 8, dtype=torch.bfloat16)
    for off in (0, 8):  # whole 16 bytes
        t = base[off:off + 512].view(4, 2, 64)
        assert at._aligned(t) is t
    for off in (1, 4):
        t = base[off:off + 512].view(4, 2, 64)
        assert t.is_contiguous() and at._aligned(t).data_ptr() % 16 == 0 and torch.equal(at._aligned(t), t)
