"""``scatter_shifted`` through the CPython binding against its general path, on the GPU:
the same bytes and flags for every form of call the binding takes, and the general path
(nothing launched by the binding) for every form it leaves."""

from __future__ import annotations

from types import SimpleNamespace

import numpy as np
import pytest
import torch

from marathon_amd import _lib, shift_kernels
from marathon_amd.shift_kernels import inv_freq_for, rope_shift, scatter_shifted
from tests.helpers import bits, randn

pytestmark = pytest.mark.gpu

BS, HEADS, D, N, BLOCKS = 16, 8, 64, 37, 9


class Sub(torch.Tensor):
    pass


def _make(gpu, dtype, hnd, form):
    """``(args, kwargs, taken)`` of one call; ``taken``: the binding launches it."""
    gen = torch.Generator().manual_seed(3)
    src = randn((N, HEADS, 2 * D), dtype, gen).to(gpu)
    shape = (BLOCKS, HEADS, BS, 2 * D) if hnd else (BLOCKS, BS, HEADS, 2 * D)
    kv = randn(shape, dtype, gen).to(gpu)
    slots = torch.randperm(BLOCKS * BS, generator=gen)[:N].to(gpu)
    shift = rope_shift(-186, D, inv_freq_for(D, 1e6), gpu)
    scale = torch.tensor([0.05], device=gpu) if dtype == torch.float8_e4m3fn else None
    flags, taken = None, True
    if form == "half rotary, flags, a bad slot":
        shift = rope_shift(7, D, inv_freq_for(D, 1e6, 0.5), gpu)
        flags = torch.zeros(1, dtype=torch.int32, device=gpu)
        slots[3] = BLOCKS * BS + 5
    elif form == "delta 0":
        shift, scale = rope_shift(0, D, inv_freq_for(D, 1e6), gpu), None
    elif form == "no shift":
        shift, scale = None, None
    elif form == "strided rows":
        src = torch.cat((src, src), dim=1)[:, :HEADS]
        kv = torch.cat((kv, kv), dim=0)[1:BLOCKS + 1]
    elif form == "the reference's RopeShift":
        shift = SimpleNamespace(delta=shift.delta, cos=shift.cos, sgn=shift.sgn,
                                emb_cos=shift.emb_cos)
    elif form == "int32 slots":
        slots, taken = slots.to(torch.int32), False
    elif form == "host slots":
        slots, taken = slots.cpu(), False
    elif form == "strided slots":
        slots, taken = torch.stack((slots, slots), dim=1)[:, 0], False
    elif form == "host tables":
        shift, taken = rope_shift(-186, D, inv_freq_for(D, 1e6), "cpu"), False
    elif form == "a subclass":
        src, taken = src.as_subclass(Sub), False
    elif form == "a number as scale":
        taken = scale is None
        scale = 0.05
    return (src, kv, slots, BS, hnd, shift), dict(k_scale=scale, error_flags=flags), taken


FORMS = ["usual", "half rotary, flags, a bad slot", "delta 0", "no shift", "strided rows",
         "the reference's RopeShift", "int32 slots", "host slots", "strided slots", "host tables",
         "a subclass", "a number as scale"]


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("hnd", [True, False])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32,
                                   torch.float8_e4m3fn])
def test_binding_and_general_path_agree(gpu, dtype, hnd, form, monkeypatch):
    print(f"case binding {dtype} hnd={hnd} {form}", flush=True)
    args, kw, taken = _make(gpu, dtype, hnd, form)
    before = args[1].clone()
    rc = _lib.binding().scatter(*args, kw["k_scale"], kw["error_flags"])
    torch.cuda.synchronize(gpu)
    assert rc == (0 if taken else None)
    assert taken or torch.equal(args[1].view(torch.uint8), before.view(torch.uint8))
    scatter_shifted(*args, **kw)
    torch.cuda.synchronize(gpu)
    got, raised = bits(args[1]), None if kw["error_flags"] is None else int(kw["error_flags"][0])
    args, kw, _ = _make(gpu, dtype, hnd, form)
    monkeypatch.setattr(shift_kernels, "_usual_call", lambda *a: None)
    scatter_shifted(*args, **kw)
    torch.cuda.synchronize(gpu)
    assert np.array_equal(got, bits(args[1]))
    assert raised == (None if kw["error_flags"] is None else int(kw["error_flags"][0]))


def test_binding_leaves_errors_to_the_general_path(gpu):
    args, _, _ = _make(gpu, torch.bfloat16, True, "usual")
    src, kv, slots, bs, hnd, shift = args
    wrong = rope_shift(5, 2 * D, inv_freq_for(2 * D, 1e6), gpu)
    for bad, err in (((src, kv, slots[:-1], bs, hnd, shift), ValueError),
                     ((src.half(), kv, slots, bs, hnd, shift), TypeError),
                     ((src, kv, slots, bs, hnd, wrong), ValueError),
                     ((src[..., ::2], kv[..., :D], slots, bs, hnd, shift), ValueError),
                     ((src, kv.cpu(), slots, bs, hnd, shift), RuntimeError)):
        assert _lib.binding().scatter(*bad, None, None) is None
        with pytest.raises(err):
            scatter_shifted(*bad)
    with pytest.raises(_lib.KVShiftError):  # the library's own refusal, through the binding
        scatter_shifted(src, kv, slots, 0, hnd, shift)
    scatter_shifted(src[:0], kv, slots[:0], bs, hnd, shift)  # nothing to move


def test_binding_launches_on_the_current_stream(gpu):
    args, kw, _ = _make(gpu, torch.bfloat16, True, "usual")
    want = args[1].clone()
    scatter_shifted(args[0], want, *args[2:])
    kv = args[1].clone()
    torch.cuda.synchronize(gpu)
    side = torch.cuda.Stream(gpu)
    with torch.cuda.stream(side):
        torch.cuda._sleep(1_000_000)  # the kernel can only have run behind this
        scatter_shifted(args[0], kv, *args[2:])
        done = torch.cuda.Event()
        done.record()
    done.synchronize()
    assert torch.equal(kv.view(torch.int16), want.view(torch.int16))
