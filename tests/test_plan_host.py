"""The plan made on the host (``mkv_plan_host``) against a per-token restatement of the
plan pass's rules, on the CPU: every record, every rotated span's table and the flags, over
the addressing modes, block sizes that are and are not powers of two, indices out of range
on either side, bad groups, negative counts, and totals that the spans do not fill or
overflow."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from marathon_amd import _lib

REC = np.dtype([("src_off", "<i8"), ("dst_off", "<i8"), ("span", "<i4"), ("delta", "<i4"),
                ("src_base", "<i4"), ("dst_base", "<i4")])
EB, LAYERS, ROT = 2, 3, 32


def _row(side, pos, index):
    """Byte offset of a token on one side (None: out of range), one token at a time."""
    bs = side["bs"]
    if side["mode"] == _lib.MKV_ADDR_TABLE:
        if pos < 0:
            return None
        ti = index + pos // bs
        if not 0 <= ti < len(side["index"]):
            return None
        blk, off = int(side["index"][ti]), pos % bs
        if not 0 <= blk < side["cap"] // bs:
            return None
    else:
        slot = pos
        if side["mode"] == _lib.MKV_ADDR_SLOTS:
            if not 0 <= index < len(side["index"]):
                return None
            slot = int(side["index"][index])
        if not 0 <= slot < side["cap"]:
            return None
        blk, off = slot // bs, slot % bs
    return (blk * side["bstride"] + off * side["ostride"]) * EB


def _side(rng, mode, bs, groups, uniform):
    blocks = int(rng.integers(4, 12))
    cap = blocks * bs + (int(rng.integers(0, bs)) if mode == _lib.MKV_ADDR_FLAT else 0)
    n = int(rng.integers(3, 40))
    index = None
    if mode == _lib.MKV_ADDR_TABLE:  # some ids out of range
        index = rng.integers(-1, blocks + 1, n).astype(np.int32)
    elif mode == _lib.MKV_ADDR_SLOTS:
        index = rng.integers(-2, cap + 2, 6 * n).astype(np.int64)
    caps = np.full(groups, cap, np.int64)
    if not uniform:
        caps -= rng.integers(0, cap // 2, groups)
    return dict(mode=mode, bs=bs, cap=cap, caps=caps, uniform=uniform, groups=groups, index=index,
                bstride=int(rng.integers(1, 9)) * 512, ostride=int(rng.integers(0, 5)) * 64)


def _fill(out, side):
    out.mode, out.block_size, out.groups, out.num_slots = (side["mode"], side["bs"],
                                                          side["groups"], side["cap"])
    out.block_stride, out.offset_stride, out.head_stride = side["bstride"], side["ostride"], 64
    if side["index"] is not None:
        out.index, out.index_len = side["index"].ctypes.data, side["index"].size
    if not side["uniform"]:
        out.group_slots = side["caps"].ctypes.data


@pytest.mark.parametrize("src_mode", range(3))
@pytest.mark.parametrize("dst_mode", range(3))
@pytest.mark.parametrize("bs", [1, 16, 24])
def test_host_plan_matches_the_rules(src_mode, dst_mode, bs):
    lib = _lib.lib()
    inv = (1.0 / (1e4 ** (np.arange(0, ROT, 2, dtype=np.float32) / ROT))).astype(np.float32)
    for seed in range(12):
        rng = np.random.default_rng(1000 * src_mode + 100 * dst_mode + 10 * bs + seed)
        groups = int(rng.integers(1, 4))
        src = _side(rng, src_mode, bs, groups, seed % 2 == 0)
        dst = _side(rng, dst_mode, 16 if bs == 1 else bs, 1, True)
        spans = np.zeros(int(rng.integers(1, 7)), _lib.SPAN_DTYPE)
        for sp in spans:
            sp["src_pos"], sp["dst_pos"] = rng.integers(-3, 60, 2)
            sp["src_index"], sp["dst_index"] = rng.integers(-1, 6, 2)
            sp["n_tokens"] = rng.choice([0, 1, 15, 16, 17, 50, -1])
            sp["delta"] = rng.choice([0, 7, -186, 2**31 - 1])
            sp["src_group"] = rng.integers(0, groups) if rng.random() < 0.8 else groups
        if seed == 3:  # positions at the end of the integer range
            spans["src_pos"][0] = spans["dst_pos"][0] = 2**63 - 5
        held = int(np.maximum(spans["n_tokens"], 0).sum())
        total = max(1, held + int(rng.choice([0, 0, 5, -3])))
        d = _lib.ShiftDesc()
        d.spans, d.n_spans, d.total_tokens = spans.ctypes.data, len(spans), total
        d.layers, d.heads, d.head_size, d.rotary, d.dtype = LAYERS, 2, 64, ROT, _lib.MKV_BF16
        d.inv_freq = inv.ctypes.data
        _fill(d.src, src)
        _fill(d.dst, dst)
        need = lib.mkv_shift_workspace_size(total, len(spans), ROT)
        room = np.full(need + 64, 0xAB, np.uint8)
        at = -room.ctypes.data % 16
        d.workspace, d.workspace_bytes = room.ctypes.data + at, need
        flags = ctypes.c_int32(-1)
        assert lib.mkv_plan_host(ctypes.byref(d), ctypes.addressof(flags)) == _lib.MKV_OK
        got = room[at:at + need]
        assert (room[at + need:] == 0xAB).all()  # nothing past the workspace
        recs = got[need - REC.itemsize * total:].view(REC)
        tables = got[:len(spans) * 8 * ROT].view(np.float32).reshape(len(spans), 2, ROT)

        want = np.zeros(total, REC)
        want["span"] = -1
        raised, g = 0, 0
        for s, sp in enumerate(spans.tolist()):
            spos, dpos, sidx, didx, n, delta, sg, dg = sp
            ok = 0 <= sg < groups and dg == 0
            raised |= 0 if ok and n >= 0 else _lib.MKV_FLAG_SPAN
            for i in range(max(n, 0)):
                if g >= total:
                    raised |= _lib.MKV_FLAG_SPAN
                    break
                if ok:
                    a = _row({**src, "cap": int(src["caps"][sg])}, spos + i if spos + i < 2**63
                             else -1, sidx + (i if src_mode == _lib.MKV_ADDR_SLOTS else 0))
                    b = _row(dst, dpos + i if dpos + i < 2**63 else -1,
                             didx + (i if dst_mode == _lib.MKV_ADDR_SLOTS else 0))
                    raised |= _lib.MKV_FLAG_SRC_RANGE if a is None else 0
                    raised |= _lib.MKV_FLAG_DST_RANGE if b is None else 0
                    if a is not None and b is not None:
                        want[g] = (a, b, s, delta, sg * LAYERS, dg * LAYERS)
                g += 1
        assert np.array_equal(recs, want), (src_mode, dst_mode, bs, seed)
        assert flags.value == raised
        for s in set(want["span"][want["delta"] != 0].tolist()) - {-1}:
            table = _lib.rope_tables([int(spans["delta"][s])], inv, ROT)[0]
            assert np.array_equal(tables[s].view(np.uint32), table.view(np.uint32))


def test_host_plan_checks_its_arguments():
    lib = _lib.lib()
    assert lib.mkv_plan_host(None, None) == _lib.MKV_ERR_ARG
    spans = np.zeros(1, _lib.SPAN_DTYPE)
    spans["n_tokens"] = 4
    room = np.zeros(512, np.uint8)
    d = _lib.ShiftDesc()
    d.spans, d.n_spans, d.total_tokens, d.layers = spans.ctypes.data, 1, 4, 1
    d.heads, d.head_size, d.dtype = 2, 64, _lib.MKV_BF16
    for side in (d.src, d.dst):
        side.mode, side.block_size, side.groups, side.num_slots = _lib.MKV_ADDR_FLAT, 1, 1, 8
        side.block_stride = 128
    at = room.ctypes.data + -room.ctypes.data % 16
    assert lib.mkv_plan_host(ctypes.byref(d), None) == _lib.MKV_ERR_ARG  # no workspace
    d.workspace, d.workspace_bytes = at, 127
    assert lib.mkv_plan_host(ctypes.byref(d), None) == _lib.MKV_ERR_ARG
    d.workspace, d.workspace_bytes = at + 8, 128
    assert lib.mkv_plan_host(ctypes.byref(d), None) == _lib.MKV_ERR_ALIGN
    d.workspace = at
    assert lib.mkv_plan_host(ctypes.byref(d), None) == _lib.MKV_OK
    d.order = _lib.MKV_ORDER_DST_PAGE  # span order only, planned or launched
    assert lib.mkv_plan_host(ctypes.byref(d), None) == _lib.MKV_ERR_UNSUPPORTED
    for side in (d.src, d.dst):
        side.k_base = side.v_base = 1 << 24
    assert lib.mkv_shift_spans_planned(ctypes.byref(d), None) == _lib.MKV_ERR_UNSUPPORTED
    d.order = _lib.MKV_ORDER_NONE
    d.workspace = None
    assert lib.mkv_shift_spans_planned(ctypes.byref(d), None) == _lib.MKV_ERR_ARG
    d.src.mode = 9
    assert lib.mkv_plan_host(ctypes.byref(d), None) == _lib.MKV_ERR_ARG
