"""Where ``ShiftPlan`` leaves the direct path by itself: on both sides of the line, in rows
and in bytes, the plan's bytes are those of either path asked for."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from marathon_amd.spans import (DIRECT_MAX_BYTES, DIRECT_MAX_TOKEN_LAYERS, CacheSet, ShiftPlan,
                                span_array)
from tests.helpers import bits, inv_freq

pytestmark = pytest.mark.gpu


def _line(dtype, heads, d, layers):
    """The most tokens the direct path takes by itself."""
    eb = torch.empty(0, dtype=dtype).element_size()
    most = DIRECT_MAX_BYTES.get(eb, DIRECT_MAX_BYTES[None])
    return min(DIRECT_MAX_TOKEN_LAYERS // layers, most // (layers * heads * 2 * d * eb))


@pytest.mark.parametrize("past", [0, 1])
@pytest.mark.parametrize("dtype,heads,d,layers", [
    (torch.float8_e4m3fn, 8, 128, 40), (torch.float8_e4m3fn, 16, 256, 24),
    (torch.bfloat16, 8, 128, 40), (torch.bfloat16, 16, 256, 28), (torch.float32, 8, 128, 40)])
def test_both_sides_of_the_line(gpu, dtype, heads, d, layers, past):
    n = _line(dtype, heads, d, layers) + past
    print(f"case direct rule {dtype} heads={heads} d={d} layers={layers} n={n}", flush=True)
    gen = torch.Generator(device=gpu).manual_seed(n)
    blocks = -(-(n + 20) // 16)

    def cache(shape):
        return torch.randn(shape, device=gpu, generator=gen).to(dtype)

    src = CacheSet([[cache((n + 5, heads, 2 * d)) for _ in range(layers)]], "flat")
    out = [torch.zeros(blocks, heads, 16, 2 * d, device=gpu).to(dtype) for _ in range(layers)]
    dst = CacheSet([out], "hnd", 16)
    table = np.random.default_rng(n).permutation(blocks).astype(np.int32)
    cut = n // 3
    spans = span_array([(3, 5, 0, 0, cut, -186, 0, 0), (3 + cut, 5 + cut, 0, 0, n - cut, 7, 0, 0)])
    kw = dict(inv_freq=inv_freq(d), src_mode="flat", dst_mode="table",
              dst_index=torch.from_numpy(table),
              k_scale=torch.full((layers,), 0.05) if dtype == torch.float8_e4m3fn else None)
    got = []
    for direct in (None, True, False):
        plan = ShiftPlan(spans, src, dst, direct=direct, **kw)
        assert plan.direct == (direct if direct is not None else past == 0)
        for t in out:
            t.zero_()
        plan.launch()
        torch.cuda.synchronize(gpu)
        got.append([bits(t) for t in out])
    for a, b, c in zip(*got):
        assert np.array_equal(a, b) and np.array_equal(a, c)
