"""When a launch waits for the copies it reads (``spans._Uploads``), on the CPU with stand-ins
for streams and events: a stream is ordered after them once, by waiting, and skipping the
waits (a capture) does not count."""

from __future__ import annotations

import weakref

import pytest
import torch

from marathon_amd import spans

BUILD, OTHER, THIRD = 0x10, 0x20, 0x30


class FakeStream:
    def __init__(self, handle, device=None):
        self.handle = handle

    def wait_stream(self, other):
        LOG.append((self.handle, "stream", other.handle))

    def wait_event(self, event):
        LOG.append((self.handle, "event", event))


class FakeTensor:
    def __init__(self):
        self.streams = set()

    def record_stream(self, stream):
        self.streams.add(stream.handle)


class FakeSet:
    def __init__(self, name, stream):
        self.name, self.upload_stream, self.blob = name, stream, FakeTensor()

    def device_tables(self, device):
        return 1, 2, None, self.name, self.blob


LOG: list = []


@pytest.fixture
def streams(monkeypatch):
    state = {"capturing": False}
    LOG.clear()
    monkeypatch.setattr(spans, "current_stream", lambda device: BUILD)
    monkeypatch.setattr(torch.cuda, "ExternalStream", FakeStream)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: state["capturing"])
    return state


def test_a_captured_launch_does_not_count_as_ordered(streams):
    own = [FakeTensor()]
    up = spans._Uploads("dev", (FakeSet("src", BUILD), FakeSet("dst", BUILD)), own)
    assert up.synced == {BUILD}  # copied there: nothing to wait for
    streams["capturing"] = True
    up.order(OTHER)
    assert LOG == [] and OTHER not in up.synced and own[0].streams == {OTHER}
    streams["capturing"] = False  # its next eager launch has to wait
    up.order(OTHER)
    assert LOG == [(OTHER, "stream", BUILD), (OTHER, "event", "src"), (OTHER, "event", "dst")]
    assert up.synced == {BUILD, OTHER}


def test_a_plan_waits_for_tables_another_stream_uploaded(streams, monkeypatch):
    """A plan built on one stream over cache sets whose base addresses went up on another:
    its launches on the build stream wait for those."""
    monkeypatch.setattr(spans._Staging, "upload",
                        lambda self, device: torch.zeros(max(self.size, 256), dtype=torch.uint8))
    monkeypatch.setattr(torch.cuda, "current_device", lambda: None)  # the CPU's index
    monkeypatch.setattr(torch.Tensor, "record_stream", lambda self, s: None)
    launched = []

    class Lib:
        def mkv_shift_spans(self, desc, stream):
            launched.append(stream.value)
            LOG.append("launch")
            return 0

    caches = [torch.zeros(32, 8, 128, dtype=torch.bfloat16) for _ in range(2)]
    sets = [spans.CacheSet([[t]], "flat") for t in caches]
    for cs, at in zip(sets, (BUILD, OTHER)):
        cs.upload_stream = at
        monkeypatch.setattr(cs, "device_tables", lambda device, at=at: (1, 2, None, at, caches[0]))
    plan = spans.ShiftPlan(spans.span_array([(0, 0, 0, 0, 5, 0, 0, 0)]), *sets, inv_freq=None,
                           dst_mode="flat", direct=True)
    monkeypatch.setattr(spans._lib, "lib", Lib)
    plan.launch()
    assert launched == [BUILD] and (BUILD, "event", OTHER) in LOG[:LOG.index("launch")]
    LOG.clear()
    plan.launch()  # ordered once
    assert LOG == ["launch"]


def test_base_tables_live_as_long_as_launches_on_other_streams(streams):
    """The tables belong to the stream that uploaded them: freed there, their memory is
    handed on in that stream's order, so every other stream that launches is recorded."""
    own = [FakeTensor()]
    sets = (FakeSet("src", BUILD), FakeSet("dst", THIRD))
    up = spans._Uploads("dev", sets, own)
    for stream in (BUILD, OTHER):
        assert stream not in up.synced
        up.order(stream)
    assert [cs.blob.streams for cs in sets] == [{BUILD, OTHER}] * 2
    assert up.synced == {BUILD, OTHER}


def test_a_captured_copy_keeps_its_host_buffer(streams):
    """A graph copies from the host buffer at each replay: the runner keeps it."""
    runner = object.__new__(spans.SmallShifts)
    runner.device, runner._captured = torch.device("cpu"), []
    for capturing in (False, True):
        streams["capturing"] = capturing
        host = torch.arange(8, dtype=torch.uint8)
        alive = weakref.ref(host)
        assert torch.equal(runner._upload(host, OTHER), host)
        del host
        assert (alive() is not None) == capturing
