"""``scatter_shifted`` on both sides of every line where its passes per wave change.

A one-layer launch makes one, two or four passes a wave by the waves it would have at one
pass (3,072, 8,192 and 12,288 of them, or 16,384 for fp8 with whole tokens per wave).
Byte for byte against the oracle, with an odd row left over in the last wave.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from marathon_amd import rope_shift, scatter_shifted
from oracle import kvshift_oracle as orc
from tests.helpers import bits, dname, inv_freq, randn

pytestmark = pytest.mark.gpu

BF16, FP32, FP8 = torch.bfloat16, torch.float32, torch.float8_e4m3fn

# (dtype, heads, head size): whole tokens per wave, tokens in segments, several tokens a wave
GEOMETRY = [(BF16, 8, 128), (BF16, 16, 256), (BF16, 3, 128), (FP32, 8, 128), (FP8, 8, 128),
            (FP8, 1, 128)]


@pytest.mark.parametrize("waves", [3072, 8192, 12288, 16384])
@pytest.mark.parametrize("dtype,heads,d", GEOMETRY)
def test_each_side_of_the_lines(gpu, dtype, heads, d, waves):
    rows_per_wave = 64 // (d * torch.empty(0, dtype=dtype).element_size() // 16)
    gen = torch.Generator().manual_seed(waves + heads)
    most = waves * rows_per_wave // heads  # tokens that make at most `waves` waves
    bs, delta, inv = 16, -566, inv_freq(d)
    nblocks = -(-(most + 1) // bs) + 3
    src = randn((most + 1, heads, 2 * d), dtype, gen, 0.05)
    kv = randn((nblocks, heads, bs, 2 * d), dtype, gen, 0.05)
    table = torch.randperm(nblocks, generator=gen)
    pos = torch.arange(3, 3 + most + 1)
    slots = table[pos // bs] * bs + pos % bs
    want = bits(kv)
    orc.scatter_shifted(bits(src), want, slots.numpy(), bs, True, delta, inv.numpy(),
                        dname(dtype), **({"k_scale": 0.05} if dtype == FP8 else {}))
    shift = rope_shift(delta, d, inv, gpu)
    src_dev, slots_dev = src.to(gpu), slots.to(gpu)
    for n in (most, most + 1):
        print(f"passes {dname(dtype)} heads={heads} d={d} n={n} waves={waves}", flush=True)
        kv_dev = kv.to(gpu)
        flags = torch.zeros(1, dtype=torch.int32, device=gpu)
        scatter_shifted(src_dev[:n], kv_dev, slots_dev[:n], bs, True, shift, error_flags=flags,
                        k_scale=0.05 if dtype == FP8 else None)
        got = bits(kv_dev)
        assert int(flags) == 0
        if n == most:  # the last token's row is still the cache's own
            last = int(slots[-1])
            ref = want.copy()
            ref[last // bs, :, last % bs] = bits(kv)[last // bs, :, last % bs]
        else:
            ref = want
        bad = int((got != ref).sum())
        assert bad == 0, f"n={n}: {bad} elements differ"
