"""The plan pass's records and tables against the host's (``mkv_plan_host``, itself held to
a per-token restatement on the CPU), on the GPU: span counts around the 64 that a wave's
lanes hold, empty spans among them, token counts around a wave and a workgroup, every
addressing mode, block sizes that are and are not powers of two, and indices out of range,
with the flags."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from marathon_amd import _lib
from marathon_amd.spans import CacheSet, ShiftPlan
from tests.helpers import inv_freq

pytestmark = pytest.mark.gpu

D, HEADS, LAYERS = 64, 2, 2


def _side(gpu, rng, mode, bs, groups):
    """``(CacheSet, host index)``; flat groups of unequal sizes, some indices out of range."""
    if mode == "flat":
        caches = [[torch.zeros(700 + 9 * g, HEADS, 2 * D, dtype=torch.bfloat16, device=gpu)
                   for _ in range(LAYERS)] for g in range(groups)]
        return CacheSet(caches, "flat"), None
    blocks = 50
    cs = CacheSet([[torch.zeros(blocks, bs, HEADS, 2 * D, dtype=torch.bfloat16, device=gpu)
                    for _ in range(LAYERS)]], "nhd", bs)
    if mode == "table":
        return cs, rng.integers(-1, blocks + 1, 90).astype(np.int32)
    return cs, rng.integers(-2, blocks * bs + 2, 1500).astype(np.int64)


@pytest.mark.parametrize("n_spans,most", [(1, 63), (1, 65), (3, 300), (63, 20), (64, 20), (65, 20)])
@pytest.mark.parametrize("src_mode,dst_mode,bs", [("flat", "table", 16), ("table", "slots", 16),
                                                  ("table", "table", 24), ("slots", "flat", 16)])
@pytest.mark.parametrize("ordered", [False, True])
def test_records_match_the_host_plan(gpu, n_spans, most, src_mode, dst_mode, bs, ordered):
    print(f"case plan pass {n_spans} spans {src_mode}->{dst_mode} bs={bs} {ordered}", flush=True)
    rng = np.random.default_rng(n_spans + most + bs)
    groups = 3 if src_mode == "flat" else 1
    src, si = _side(gpu, rng, src_mode, bs, groups)
    dst, di = _side(gpu, rng, dst_mode, bs, 1)
    spans = np.zeros(n_spans, _lib.SPAN_DTYPE)
    for sp in spans:
        sp["src_pos"], sp["dst_pos"] = rng.integers(-2, 500, 2)
        sp["src_index"], sp["dst_index"] = rng.integers(-1, 30, 2)
        sp["n_tokens"] = most if n_spans == 1 else rng.choice([0, 1, most, most // 2])
        sp["delta"] = rng.choice([0, 186, -3000])
        sp["src_group"] = rng.integers(0, groups + (rng.random() < 0.1))
    if not spans["n_tokens"].any():
        spans["n_tokens"][-1] = 5
    total = int(spans["n_tokens"].sum())
    inv = inv_freq(D)
    plan = ShiftPlan(spans, src, dst, inv_freq=inv, src_mode=src_mode, src_index=si,
                     dst_mode=dst_mode, dst_index=di, direct=False, order="none")
    (d,) = plan.descs
    order = rng.permutation(total).astype(np.int32)
    if ordered:
        order[0] = total + 3 if total > 1 else order[0]  # one entry out of range: not moved
        held = torch.from_numpy(order).to(gpu)
        d.token_order = held.data_ptr()
    flags = torch.zeros(1, dtype=torch.int32, device=gpu)
    plan.launch(error_flags=flags)
    torch.cuda.synchronize(gpu)

    h = _lib.ShiftDesc()
    ctypes.memmove(ctypes.byref(h), ctypes.byref(d), ctypes.sizeof(d))
    h.token_order, h.spans, h.inv_freq = None, spans.ctypes.data, inv.data_ptr()
    for side, cs, index in ((h.src, src, si), (h.dst, dst, di)):
        side.index = None if index is None else index.ctypes.data
        caps, uniform = cs.base_tables()[2], cs.base_tables()[4]
        side.group_slots = None if uniform else caps.ctypes.data
    need = _lib.lib().mkv_shift_workspace_size(total, n_spans, D)
    room = np.zeros(need + 16, np.uint8)
    at = -room.ctypes.data % 16
    h.workspace, h.workspace_bytes = room.ctypes.data + at, need
    raised = ctypes.c_int32()
    _lib.check(_lib.lib().mkv_plan_host(ctypes.byref(h), ctypes.addressof(raised)))
    want, got = room[at:at + need], plan.workspace[:need].cpu().numpy()
    recs = want[need - 32 * total:].reshape(total, 32)
    expect = recs.copy()
    if ordered:
        empty = np.zeros(32, np.uint8)
        empty[16:20] = 0xFF  # span -1
        expect = np.stack([recs[t] if t < total else empty for t in order])
    assert np.array_equal(got[need - 32 * total:].reshape(total, 32), expect)
    tables = lambda a: a[:n_spans * 8 * D].reshape(n_spans, 8 * D)  # noqa: E731
    for s in set(recs.view(np.int32)[:, 4].tolist()) - {-1}:
        if spans["delta"][s] != 0:
            assert np.array_equal(tables(got)[s], tables(want)[s])
    if not ordered:
        assert int(flags.item()) == raised.value
