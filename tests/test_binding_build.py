"""The CPython binding as built, on the CPU: it has no thread-local storage (a TLS block that
a thread has not touched slows every other library's TLS access in it), and it leaves calls
on anything but GPU tensors to the general path."""

from __future__ import annotations

import os
import struct
import warnings
from types import SimpleNamespace

import pytest
import torch

from marathon_amd import _lib, shift_kernels

PT_TLS = 7


def test_binding_has_no_tls_segment():
    with open(os.path.join(_lib.LIB_DIR, "marathon_binding.so"), "rb") as f:
        elf = f.read()
    assert elf[:5] == b"\x7fELF\x02"
    at, = struct.unpack_from("<Q", elf, 32)  # e_phoff
    size, count = struct.unpack_from("<HH", elf, 54)  # e_phentsize, e_phnum
    assert PT_TLS not in [struct.unpack_from("<I", elf, at + k * size)[0] for k in range(count)]


def test_binding_leaves_other_calls():
    scatter = _lib.binding().scatter
    src, kv = torch.zeros(2, 8, 128), torch.zeros(4, 8, 16, 128)
    slots = torch.zeros(2, dtype=torch.int64)
    assert scatter(src, kv, slots, 16, True, None, None, None) is None
    assert scatter(None, 3, "x", 16, True, None, None, None) is None


@pytest.mark.parametrize("what", ["header", "torch"])
def test_a_module_built_for_something_else_is_refused(monkeypatch, what):
    """The module calls the library and torch by the headers it was compiled with."""
    _lib.binding()
    monkeypatch.setattr(_lib, "_BINDING", None)
    if what == "header":
        monkeypatch.setattr(_lib, "MKV_ABI_VERSION", _lib.MKV_ABI_VERSION + 1)
    else:
        monkeypatch.setattr(torch, "__version__", "0.0.1")
    with pytest.raises(RuntimeError, match="rebuild"):
        _lib.binding()
    monkeypatch.undo()
    assert _lib.binding().scatter is not None


def test_scatter_shifted_does_without_the_module(monkeypatch):
    """The general path needs only the library: with no module it takes every call, after
    one warning."""
    monkeypatch.setattr(shift_kernels, "_usual_call", None)
    monkeypatch.setattr(_lib, "_BINDING", None)
    monkeypatch.setattr(_lib, "LIB_DIR", "/nonexistent")
    args = (torch.zeros(2, 8, 128), torch.zeros(4, 8, 16, 128), torch.zeros(2, dtype=torch.int64),
            16, True, None)
    with pytest.warns(RuntimeWarning, match="marathon_binding.so"):
        with pytest.raises(RuntimeError, match="not on a HIP device"):
            shift_kernels.scatter_shifted(*args)
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        with pytest.raises(RuntimeError, match="not on a HIP device"):
            shift_kernels.scatter_shifted(*args)


def test_warmup_loads_what_the_first_call_needs(monkeypatch):
    monkeypatch.setattr(shift_kernels, "_usual_call", None)
    shift_kernels.warmup(SimpleNamespace(is_cuda=False), 16, True)
    assert shift_kernels._usual_call is None
    shift_kernels.warmup(SimpleNamespace(is_cuda=True), 16, True)
    assert shift_kernels._usual_call is _lib.binding().scatter
