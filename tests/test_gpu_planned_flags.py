"""The error flags of a ``SmallShifts`` step planned on the host, on the GPU: every launch that
is given ``error_flags`` raises them, in its first word as the kernels do, and moves the same
rows as one without."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from marathon_amd import _lib
from marathon_amd.spans import CacheSet, SmallShifts
from tests.helpers import inv_freq

pytestmark = pytest.mark.gpu


def _bad_step(gpu):
    """A runner and a step planned on the host: a destination block that does not exist."""
    src = CacheSet([[torch.ones(100, 8, 128, dtype=torch.bfloat16, device=gpu)]], "flat")
    dst = CacheSet([[torch.zeros(9, 8, 16, 128, dtype=torch.bfloat16, device=gpu)]], "hnd", 16)
    runner = SmallShifts(src, dst, inv_freq=inv_freq(64), src_mode="flat", dst_mode="table")
    table = np.concatenate((np.arange(1, 8), [99], np.zeros(65))).astype(np.int32)
    return runner, ([(0, 0, 0, 0, 100, 7, 0, 0), (5, 112, 0, 0, 16, 7, 0, 0)], None, table)


def test_flags_of_a_planned_step_go_into_one_word(gpu):
    print("case planned flags, one word", flush=True)
    runner, step = _bad_step(gpu)
    words = torch.zeros(3, 2, dtype=torch.int32, device=gpu)
    runner.run(*step, error_flags=words[1:])
    assert not runner._last and runner._now is runner.desc
    want = torch.zeros_like(words)
    want[1, 0] = _lib.MKV_FLAG_DST_RANGE
    assert torch.equal(words, want)


@pytest.mark.parametrize("given", [False, True])
def test_a_relaunch_raises_the_flags_again(gpu, given):
    print(f"case planned flags, relaunch {given}", flush=True)
    runner, step = _bad_step(gpu)
    out = runner.dst.caches[0][0]
    first = torch.zeros(1, dtype=torch.int32, device=gpu)
    runner.run(*step, error_flags=first if given else None)
    moved = out.clone()
    assert int(moved.any(-1).sum()) == 100 * 8  # the first span's rows, and no other
    for stream in (None, torch.cuda.current_stream(gpu).cuda_stream):
        out.zero_()
        again = torch.zeros(1, dtype=torch.int32, device=gpu)
        runner.launch(stream, error_flags=again)
        assert again.item() == _lib.MKV_FLAG_DST_RANGE
        assert torch.equal(out, moved)
    out.zero_()
    runner.launch()  # nobody asks
    assert torch.equal(out, moved)
    assert first.item() == (_lib.MKV_FLAG_DST_RANGE if given else 0)
    good = (step[0][:1], None, step[2])
    runner.run(*good, error_flags=again.zero_())  # the next step's flags are its own
    assert again.item() == 0
