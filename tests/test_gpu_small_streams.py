"""``SmallShifts`` on another stream than the one that uploaded the caches' base addresses and
the runner's frequencies, on the GPU: the uploads are held behind a sleep on their stream, and
a step in each of the three forms -- in the launch, planned on the host, staged for the plan
pass -- run at once on a second stream moves what it moves on one stream."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from marathon_amd.spans import CacheSet, SmallShifts
from tests.helpers import bits, inv_freq, randn

pytestmark = pytest.mark.gpu

HEADS, D, BS, LAYERS = 16, 64, 16, 2


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("form,tokens", [("launch", 40), ("planned", 300), ("staged", 2000)])
def test_steps_wait_for_uploads_on_another_stream(gpu, form, tokens, dtype):
    print(f"case small streams {form} {dtype}", flush=True)
    gen = torch.Generator().manual_seed(tokens)
    blocks = -(-tokens // BS) + 1
    src = [randn((tokens, HEADS, 2 * D), dtype, gen).to(gpu) for _ in range(LAYERS)]
    out = [torch.zeros(blocks, HEADS, BS, 2 * D, device=gpu).to(dtype) for _ in range(LAYERS)]
    table = torch.randperm(blocks, generator=gen).numpy().astype(np.int32)
    if form != "launch":  # more entries than a launch carries
        table = np.concatenate((table, np.zeros(65, np.int32)))
    rows = [(0, 3, 0, 0, tokens, 186, 0, 0)]
    scale = torch.tensor([0.031, 0.066]) if dtype == torch.float8_e4m3fn else None

    def runner():
        return SmallShifts(CacheSet([src], "flat"), CacheSet([out], "hnd", BS),
                           inv_freq=inv_freq(D), src_mode="flat", dst_mode="table", k_scale=scale)

    one = runner()
    one.run(rows, None, table)
    torch.cuda.synchronize(gpu)
    got = {"launch": bool(one._last), "planned": not one._last and one._now is one.desc,
           "staged": one._now is one.stage_desc}
    assert [k for k, v in got.items() if v] == [form]
    assert one.direct == (form != "staged")
    want = [bits(t) for t in out]
    assert any(w.any() for w in want)
    for t in out:
        t.view(torch.uint8).zero_()
    torch.cuda.synchronize(gpu)
    uploads, launches = torch.cuda.Stream(gpu), torch.cuda.Stream(gpu)
    with torch.cuda.stream(uploads):
        torch.cuda._sleep(1_000_000)
        two = runner()
    with torch.cuda.stream(launches):
        two.run(rows, None, table)
    torch.cuda.synchronize(gpu)
    for t, w in zip(out, want):
        assert np.array_equal(bits(t), w)
