"""Where the plan pass's rotation tables are made (``MKV_PLAN_TABLE_GROUPS``), on the GPU: the
build whose record workgroups make them shifts to the default build's bytes, in the span
counts and block sizes of both plan kernels, whatever the workspace held before."""

from __future__ import annotations

import ctypes
import os

import numpy as np
import pytest
import torch

from marathon_amd import _lib
from marathon_amd.spans import CacheSet, ShiftPlan, span_array
from tests.helpers import bits, inv_freq, randn

pytestmark = pytest.mark.gpu

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "_lib",
                   "libkvshift_tables_in_records.so")
HEADS, D = 8, 64


@pytest.mark.parametrize("n_spans", [1, 64, 65])
@pytest.mark.parametrize("bs", [16, 24])
def test_tables_in_record_workgroups(gpu, monkeypatch, bs, n_spans):
    print(f"case tables in records bs={bs} spans={n_spans}", flush=True)
    gen = torch.Generator().manual_seed(n_spans + bs)
    per = 5
    blocks = -(-n_spans * per // bs) + 1
    src = CacheSet([[randn((n_spans * per, HEADS, 2 * D), torch.bfloat16, gen).to(gpu)]], "flat")
    out = torch.zeros(blocks, bs, HEADS, 2 * D, dtype=torch.bfloat16, device=gpu)
    dst = CacheSet([[out]], "nhd", bs)
    table = torch.randperm(blocks, generator=gen).to(torch.int32)
    rows = [(k * per, k * per, 0, 0, per, 186 - 7 * k, 0, 0) for k in range(n_spans)]
    plan = ShiftPlan(span_array(rows), src, dst, inv_freq=inv_freq(D), dst_mode="table",
                     dst_index=table, direct=False)
    got = []
    for cdll in (_lib.lib(), _lib._bind(ctypes.CDLL(LIB, mode=ctypes.RTLD_LOCAL))):
        monkeypatch.setattr(_lib, "_LIB", cdll)
        plan.workspace.fill_(0x3F)
        out.zero_()
        plan.launch()
        torch.cuda.synchronize(gpu)
        got.append(bits(out))
    assert got[0].any()
    assert np.array_equal(*got)
