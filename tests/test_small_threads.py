"""A ``SmallShifts`` runner shared by threads, on the CPU with a stand-in for the launches: a
step that another thread starts between this one's descriptor and its launch does not get
into that launch, in any of a step's three forms."""

from __future__ import annotations

import threading

import numpy as np
import pytest
import torch

from marathon_amd import _lib, spans
from marathon_amd.spans import CacheSet, SmallShifts

TOKENS = {"launch": (7, 9), "planned": (70, 90), "staged": (700, 900)}


@pytest.mark.parametrize("form", list(TOKENS))
def test_a_launch_is_of_its_own_thread_s_step(monkeypatch, form):
    real, empty = _lib.lib(), torch.empty
    launched = {}
    busy = threading.Event()

    class Lib:
        mkv_plan_host = real.mkv_plan_host

        def __getattr__(self, name):  # the launches
            def launch(desc, stream):
                launched[threading.get_ident()] = (name, desc._obj.total_tokens)
                return 0
            return launch

    monkeypatch.setattr(spans._Staging, "upload",
                        lambda self, device: torch.zeros(max(self.size, 256), dtype=torch.uint8))
    monkeypatch.setattr(torch, "empty", lambda *a, pin_memory=False, **k: empty(*a, **k))
    monkeypatch.setattr(torch.cuda, "current_device", lambda: None)  # the CPU's index
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(spans, "current_stream", lambda device: 0x10)
    sets = [CacheSet([[torch.zeros(2000, 8, 128, dtype=torch.bfloat16)]], "flat") for _ in range(2)]
    for cs in sets:
        cs.upload_stream = 0x10
        monkeypatch.setattr(cs, "device_tables", lambda device: (1, 2, None, None, None))
    runner = SmallShifts(*sets, inv_freq=None, src_mode="slots", dst_mode="flat")
    monkeypatch.setattr(spans._lib, "lib", Lib)
    index = np.arange(64 if form == "launch" else 2000)  # past 64 a step leaves the launch
    mine, theirs = TOKENS[form]

    def step(n):
        runner.run([(0, 0, 0, 0, n, 0, 0, 0)], index, None)

    def device_asked_for():
        if not busy.is_set():  # this thread's step has its descriptor and not its launch yet
            busy.set()
            other.start()
            other.join(0.3)

    other = threading.Thread(target=step, args=(theirs,))
    monkeypatch.setattr(torch.cuda, "current_device", device_asked_for)
    step(mine)
    other.join()
    fn = {"launch": "mkv_shift_spans_small", "planned": "mkv_shift_spans_planned",
          "staged": "mkv_shift_spans"}[form]
    assert launched[threading.get_ident()] == (fn, mine)
    assert launched[other.ident] == (fn, theirs)
