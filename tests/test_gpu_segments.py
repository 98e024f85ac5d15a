"""Tokens of more rows than one workgroup sweep, byte for byte against the oracle.

A token whose KV heads exceed the rows a workgroup covers in one sweep is cut into
segments of its own workgroups: a power of two of them or not, whole or with a remainder,
and with rows of one token per wave or several.  Every entry point that launches the shift
kernel is run: two launches, direct, small, and one layer per call.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from marathon_amd import rope_shift, scatter_shifted
from marathon_amd.spans import CacheSet, ShiftPlan, SmallShifts, span_array
from oracle import kvshift_oracle as orc
from tests.helpers import bits, dname, inv_freq, oracle_side, oracle_spans, randn

pytestmark = pytest.mark.gpu

BF16, FP16, FP32, FP8 = torch.bfloat16, torch.float16, torch.float32, torch.float8_e4m3fn

# (dtype, head size, heads): bf16 rows of 128 make sweeps of 8, of 256 sweeps of 4
CASES = [(BF16, 128, 9), (BF16, 128, 12), (BF16, 128, 16), (BF16, 128, 40), (FP16, 128, 24),
         (BF16, 256, 5), (BF16, 256, 16), (BF16, 256, 18), (BF16, 64, 17), (FP32, 128, 40),
         (FP32, 256, 16), (FP8, 128, 40), (FP8, 256, 20)]


@pytest.mark.parametrize("dtype,d,heads", CASES)
def test_segments_match_oracle(gpu, dtype, d, heads):
    gen = torch.Generator().manual_seed(heads * 1000 + d)
    layers, bs, rows = 2, 16, 150
    inv = inv_freq(d)
    scale = torch.tensor([0.05, 0.031]) if dtype == FP8 else None
    src_cpu = [randn((rows, heads, 2 * d), dtype, gen, 0.05) for _ in range(layers)]
    dst_cpu = [randn((20, heads, bs, 2 * d), dtype, gen, 0.05) for _ in range(layers)]
    table = torch.randperm(20, generator=gen).to(torch.int32)
    # one-token spans, a span that ends inside an XCD's share of the tiles, an unmoved one
    raw = [(3, 5, 0, 0, 1, 186, 0, 0), (10, 21, 0, 0, 61, -566, 0, 0),
           (90, 100, 0, 0, 7, 0, 0, 0), (100, 120, 0, 0, 50, 20000, 0, 0)]
    spans = span_array(raw)

    def sets():
        return (CacheSet([[t.to(gpu) for t in src_cpu]], "flat"),
                CacheSet([[t.to(gpu) for t in dst_cpu]], "hnd", bs))

    src, dst = sets()
    want = oracle_side(dst, "table", table)
    orc.shift_spans(oracle_spans(spans), oracle_side(src, "flat", None), want, inv.numpy(),
                    dname(dtype), k_scale=None if scale is None else scale.numpy())
    kw = dict(inv_freq=inv, src_mode="flat", dst_mode="table", k_scale=scale)

    def check(dst, what):
        torch.cuda.synchronize(gpu)
        for layer in range(layers):
            bad = int((bits(dst.caches[0][layer]) != want.caches[0][layer]).sum())
            assert bad == 0, f"{what} layer {layer}: {bad} elements differ"

    for direct in (False, True):
        print(f"segments {dname(dtype)} d={d} heads={heads} direct={direct}", flush=True)
        src, dst = sets()
        plan = ShiftPlan(spans, src, dst, dst_index=table, direct=direct, **kw)
        flags = torch.zeros(1, dtype=torch.int32, device=gpu)
        plan.launch(error_flags=flags)
        check(dst, f"direct={direct}")
        assert int(flags) == 0
    src, dst = sets()
    small = SmallShifts(src, dst, **kw)
    if small.fits(len(raw), 119):
        small.run(raw, None, table.numpy())
        check(dst, "small")
    src, dst = sets()
    for layer in range(layers):
        for sp, dp, _, _, n, delta, _, _ in raw:
            pos = torch.arange(dp, dp + n)
            slots = (table.long()[pos // bs] * bs + pos % bs).to(gpu)
            scatter_shifted(src.caches[0][layer][sp:sp + n], dst.caches[0][layer], slots, bs, True,
                            rope_shift(delta, d, inv, gpu),
                            k_scale=None if scale is None else float(scale[layer]))
    check(dst, "one layer per call")
