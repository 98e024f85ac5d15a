"""A ``SmallShifts`` step captured in a HIP graph, on the GPU: each form of a step, replayed
after eager steps of the same runner that reuse pinned memory, moves the captured rows."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from marathon_amd.spans import CacheSet, SmallShifts
from tests.helpers import bits, inv_freq, randn

pytestmark = pytest.mark.gpu

HEADS, D, BS, LAYERS = 8, 64, 16, 2


@pytest.mark.parametrize("form,tokens", [("launch", 40), ("planned", 300), ("staged", 2000)])
def test_captured_steps_replay(gpu, form, tokens):
    print(f"case small capture {form}", flush=True)
    gen = torch.Generator().manual_seed(tokens)
    blocks = -(-tokens // BS) + 1
    src = [randn((tokens, HEADS, 2 * D), torch.bfloat16, gen).to(gpu) for _ in range(LAYERS)]
    out = [torch.zeros(blocks, HEADS, BS, 2 * D, dtype=torch.bfloat16, device=gpu)
           for _ in range(LAYERS)]
    runner = SmallShifts(CacheSet([src], "flat"), CacheSet([out], "hnd", BS),
                         inv_freq=inv_freq(D), src_mode="flat", dst_mode="table")
    pad = np.zeros(0 if form == "launch" else 65, np.int32)  # more than a launch carries

    def step(seed):
        table = np.random.default_rng(seed).permutation(blocks).astype(np.int32)
        return [(0, 3, 0, 0, tokens, 186 - seed, 0, 0)], None, np.concatenate((table, pad))

    def eager(seed):
        for t in out:
            t.zero_()
        runner.run(*step(seed))
        torch.cuda.synchronize(gpu)
        return [bits(t) for t in out]

    want = eager(0)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        runner.run(*step(0))
    for replay in range(4):
        for seed in range(1, 4):
            other = eager(seed)
        for t in out:
            t.zero_()
        torch.cuda.synchronize(gpu)
        graph.replay()
        torch.cuda.synchronize(gpu)
        for t, w, o in zip(out, want, other):
            got = bits(t)
            assert np.array_equal(got, w), replay
            assert not np.array_equal(got, o)
