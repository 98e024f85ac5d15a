"""When a launch waits for the copies it reads (``spans._Uploads``), on the CPU with stand-ins
for streams and events: a stream is ordered after them once, by waiting, and skipping the
waits (a capture) does not count."""

from __future__ import annotations

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
