"""``SmallShifts`` steps past the in-launch limits against the two-launch path's bytes, on
the GPU: planned on the host up to the largest plan that is, then staged for the plan
pass; every element type, geometries the in-launch and direct paths refuse (one head,
blocks of 24), stores of unequal sizes, and an index out of range."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from marathon_amd import _lib
from marathon_amd.spans import HOST_PLAN_MAX_BYTES, CacheSet, ShiftPlan, SmallShifts, span_array
from tests.helpers import bits, inv_freq, randn

pytestmark = pytest.mark.gpu

HEAD, SPANS = 64, 3
LARGEST = (HOST_PLAN_MAX_BYTES - SPANS * 8 * HEAD) // 32  # tokens of a step planned on the host

DTYPES = [torch.bfloat16, torch.float16, torch.float32, torch.float8_e4m3fn]


@pytest.mark.parametrize("tokens", [65, LARGEST, LARGEST + 1, 2500])
@pytest.mark.parametrize("heads,bs,flat", [(8, 16, False), (1, 16, True), (8, 24, True),
                                           (16, 16, False)])
@pytest.mark.parametrize("dtype", DTYPES)
def test_planned_steps_match_the_plan_pass(gpu, dtype, heads, bs, flat, tokens):
    print(f"case planned {dtype} heads={heads} bs={bs} flat={flat} tokens={tokens}", flush=True)
    gen = torch.Generator().manual_seed(tokens + heads)
    rng = np.random.default_rng(tokens + heads)
    d, layers = HEAD, 2
    cuts = [0, tokens // 3, tokens // 3 + 1, tokens]  # SPANS spans, one of one token
    blocks = -(-(tokens + 100) // bs)
    if flat:  # a store per span, of unequal sizes
        src = CacheSet([[randn((tokens + 7 * g, heads, 2 * d), dtype, gen).to(gpu)
                         for _ in range(layers)] for g in range(3)], "flat")
    else:
        src = CacheSet([[randn((blocks, bs, heads, 2 * d), dtype, gen).to(gpu)
                         for _ in range(layers)]], "nhd", bs)
    before = [randn((blocks, heads, bs, 2 * d), dtype, gen).to(gpu) for _ in range(layers)]
    out = [t.clone() for t in before]
    dst = CacheSet([out], "hnd", bs)
    si = None if flat else rng.permutation(blocks).astype(np.int32)
    di = rng.permutation(blocks).astype(np.int32)
    di[0] = blocks + 3  # tokens of this block are flagged and not moved
    di = np.concatenate((di, np.zeros(65, np.int32)))  # more than a launch carries
    rows = [(5 + 2 * k if flat else cuts[k] + 9, cuts[k] + 40, 0, 0, cuts[k + 1] - cuts[k],
             (0, 186, -3000)[k], k if flat else 0, 0) for k in range(3)]
    scale = torch.tensor([0.031, 0.066]) if dtype == torch.float8_e4m3fn else None
    kw = dict(inv_freq=inv_freq(d), src_mode="flat" if flat else "table", dst_mode="table",
              k_scale=scale)
    flags = torch.zeros(2, dtype=torch.int32, device=gpu)
    if tokens == 65:
        rows[0] = (rows[0][0], 5, *rows[0][2:])  # into the bad block
    runner = SmallShifts(src, dst, **kw)
    assert runner.fits(len(rows), tokens)
    runner.run(rows, si, di, error_flags=flags[:1])
    assert not runner._last  # not in the launch
    assert (runner._now is runner.desc) == (tokens <= LARGEST)
    torch.cuda.synchronize(gpu)
    got = [bits(t) for t in out]
    for t, b in zip(out, before):
        t.copy_(b)
    plan = ShiftPlan(span_array(rows), src, dst, src_index=si, dst_index=di, direct=False, **kw)
    plan.launch(error_flags=flags[1:])
    torch.cuda.synchronize(gpu)
    for g, t in zip(got, out):
        assert np.array_equal(g, bits(t))
    assert flags[0].item() == flags[1].item()
    assert bool(flags[0].item() & _lib.MKV_FLAG_DST_RANGE) == (tokens == 65)
