"""Worker-side load path of the shift connector, one HIP launch per engine step.

The reference's ``MarathonShiftConnector`` (src/marathon/vllm_shift_connector.py) runs,
for every load of a step and every layer, ``ShiftStore.read`` and one
``scatter_shifted`` launch (:481-534, loop at :505-518): 40 launches per load on
Qwen3-14B, plus per-layer Python.  :class:`ShiftLoader` keeps the same inputs -- the
``_Load`` list (:135-140), the registered paged caches (:393-412) and the session store
-- and issues the whole step as one batched shift (:class:`marathon_amd.spans.ShiftPlan`,
or :class:`marathon_amd.spans.SmallShifts` for a short step): every load x every layer,
sources read straight out of each session's store buffer.

Also here, as host logic: the layout detection of ``register_kv_caches`` (:393-402) and
the multi-segment block alignment of ``_accept_multi`` (:225-245).

Slots on the device.  The reference's scheduler builds every load's and save's int64
slot list on the host (``slots()``, :349-366 / :320) and the worker copies it H2D
(:504): 8 bytes per token.  A :class:`Load` or :class:`Save` built with ``from_blocks``
carries the request's block table and a position range instead.  The kernels turn
positions into slots on the device (``MKV_ADDR_TABLE``), so the host ships 4 bytes per
16 tokens.  Either store works as the source or target: the reference's flat
:class:`~marathon_amd.shift_store.ShiftStore`, or the
:class:`~marathon_amd.block_store.BlockShiftStore` pool, read and written through its
block tables.
"""

from __future__ import annotations

import logging
import os
import time
from dataclasses import dataclass

import numpy as np
import torch

from . import _lib
from .block_store import BlockShiftStore
from .shift_store import ShiftStore, slots as host_slots
from .spans import CacheSet, ShiftPlan, SmallShifts

logger = logging.getLogger("marathon_amd.shift")

#: ``MARATHON_VERIFY_LOAD=1`` reads every loaded span back out of the paged cache and
#: compares it with torch's rotation of the same source rows, per layer, and logs the
#: error (vllm_shift_connector.py:95-102, :444-480).  Diagnostic only, off by default:
#: it reads, it never writes a cache, and the kernel still does every load.
VERIFY_LOAD = os.environ.get("MARATHON_VERIFY_LOAD", "") not in ("", "0")


def store_from_config(extra: dict | None, worker: bool, *, block_layout: bool = False,
                      block_size: int = 16):
    """The connector's store, configured as the reference's connector configures it
    (vllm_shift_connector.py:168-178): budget from ``kv_connector_extra_config``
    ``store_tokens``, else ``MARATHON_STORE_TOKENS``, else 32,768; ``store_device``;
    ``session_tokens`` (one session's positions, allocated once).  Tensors only on the
    worker; the scheduler keeps the tensor-free mirror.  ``block_layout`` returns the
    :class:`BlockShiftStore` with the reference's truncation rule instead."""
    from .shift_store import DEFAULT_STORE_TOKENS

    extra = extra or {}
    budget = int(extra.get("store_tokens", os.environ.get("MARATHON_STORE_TOKENS",
                                                          DEFAULT_STORE_TOKENS)))
    device = str(extra.get("store_device", "cuda"))
    if block_layout:
        return BlockShiftStore(budget, device, allocate=worker, block_size=block_size)
    cap = int(extra.get("session_tokens", 0) or 0)
    return ShiftStore(budget, device, allocate=worker, session_cap=cap)


def _rotate_half(x: torch.Tensor) -> torch.Tensor:
    half = x.shape[-1] // 2
    return torch.cat((-x[..., half:], x[..., :half]), dim=-1)


def _rerotate(k: torch.Tensor, delta: int, inv_freq: torch.Tensor) -> torch.Tensor:
    """torch's rotation of fp32 keys by ``delta``: the reference's ``rerotate_keys``
    (kvshift.py:44-61), here only the yardstick of the read-back check."""
    if delta == 0:
        return k
    angles = float(delta) * inv_freq.to(device=k.device, dtype=torch.float32)
    emb = torch.cat((angles, angles), dim=-1)
    return k * emb.cos() + _rotate_half(k) * emb.sin()


@dataclass
class Save:
    """One save of a step (vllm_shift_connector.py:143-151): the positions this step
    computed, ``slots`` in the paged cache, stored from ``dst_start``.

    ``Save.from_blocks`` leaves ``slots`` None: the paged rows are then positions
    ``[dst_start, dst_start + n_tokens)`` through ``block_ids``, resolved on the device.
    """

    session: str
    slots: torch.Tensor | None  # int64 [T], on the host or the GPU
    dst_start: int
    block_ids: object = None  # the request's block table (device-side slots)
    n_tokens: int = 0

    @classmethod
    def from_blocks(cls, session: str, block_ids, lo: int, hi: int) -> "Save":
        return cls(session, None, int(lo), block_ids, int(hi) - int(lo))

    @property
    def n(self) -> int:
        return int(self.slots.numel()) if self.slots is not None else max(int(self.n_tokens), 0)

    @property
    def paged_pos(self) -> int:
        return int(self.dst_start)


@dataclass
class Load:
    """One load of a step (vllm_shift_connector.py:135-140).

    ``Load.from_blocks`` leaves ``slots`` None: the destination is then positions
    ``[dst_start, dst_start + n_tokens)`` through ``block_ids``, resolved on the device.
    """

    session: str
    slots: torch.Tensor | None  # int64 [T]: destination slots of positions [lo, hi), on
    # the host or the GPU
    src_start: int  # first source position in the session's store
    delta: int
    block_ids: object = None  # the request's block table (device-side slots)
    dst_start: int = 0
    n_tokens: int = 0

    @classmethod
    def from_blocks(cls, session: str, block_ids, lo: int, hi: int, delta: int) -> "Load":
        return cls(session, None, int(lo) - int(delta), int(delta), block_ids, int(lo),
                   int(hi) - int(lo))

    @property
    def n(self) -> int:
        return int(self.slots.numel()) if self.slots is not None else max(int(self.n_tokens), 0)

    @property
    def paged_pos(self) -> int:
        return int(self.dst_start)


class _CacheSets:
    """CacheSets by role, rebuilt only when the tensors they describe change.

    A CacheSet validates every tensor and reads every base address once; a step that
    reuses the same caches should not pay that again.  Rows given as the very list
    objects of the cached set match at once; otherwise the tensors' ids are compared
    (the cached set keeps its tensors alive, so an id cannot be reused while cached).
    """

    def __init__(self, block_size: int) -> None:
        self.block_size = block_size
        self._sets: dict[str, tuple] = {}

    @staticmethod
    def _ids(rows) -> tuple | None:
        return None if rows is None else tuple(tuple(id(t) for t in row) for row in rows)

    def get(self, role: str, caches: list, layout: str, block_size: int | None = None,
            v_caches: list | None = None) -> CacheSet:
        hit = self._sets.get(role)
        if hit is not None:
            rows, v_rows, _, cs = hit
            same = len(rows) == len(caches) and all(a is b for a, b in zip(rows, caches)) and (
                v_caches is None if v_rows is None else
                v_caches is not None and len(v_rows) == len(v_caches)
                and all(a is b for a, b in zip(v_rows, v_caches)))
            if same or hit[2] == (self._ids(caches), self._ids(v_caches)):
                if not same:
                    self._sets[role] = (list(caches), None if v_caches is None else
                                        list(v_caches), hit[2], cs)
                return cs
        bs = self.block_size if block_size is None else block_size
        cs = CacheSet([list(r) for r in caches], layout, bs,
                      v_caches=None if v_caches is None else [list(r) for r in v_caches])
        self._sets[role] = (list(caches), None if v_caches is None else list(v_caches),
                            (self._ids(caches), self._ids(v_caches)), cs)
        return cs


class _SmallRunners:
    """One :class:`~marathon_amd.spans.SmallShifts` per (source set, destination set,
    modes, K scales), reused across steps while those stay the same objects."""

    def __init__(self) -> None:
        self._runners: dict[tuple, tuple] = {}

    def get(self, src: CacheSet, dst: CacheSet, src_mode: str, dst_mode: str, inv_freq,
            k_scale=None) -> SmallShifts:
        scales = None if k_scale is None else tuple(k_scale.tolist())
        key = (id(src), id(dst), src_mode, dst_mode, scales)
        hit = self._runners.get(key)
        if hit is None or hit[0] is not src or hit[1] is not dst:
            if len(self._runners) >= 16:  # caches or stores replaced many times over
                self._runners.clear()
            hit = self._runners[key] = (src, dst, SmallShifts(
                src, dst, inv_freq=inv_freq, src_mode=src_mode, dst_mode=dst_mode,
                k_scale=k_scale))
        return hit[2]


def _host(index) -> np.ndarray | None:
    if index is None or isinstance(index, np.ndarray):
        return index
    return index.numpy()


def _int32_table(t) -> np.ndarray:
    if isinstance(t, np.ndarray) and t.dtype == np.int32:
        return t.reshape(-1)
    if isinstance(t, torch.Tensor):
        return t.detach().to("cpu", torch.int32).numpy().reshape(-1)
    return np.asarray(t, dtype=np.int32).reshape(-1)


def table_window(table: np.ndarray, pos: int, n: int, block_size: int):
    """The blocks of ``table`` that positions ``[pos, pos + n)`` touch, and ``pos``
    relative to the first of them: only those entries need to reach the device."""
    k0 = pos // block_size
    k1 = -(-(pos + n) // block_size)
    if pos < 0 or k1 > table.size:
        raise ValueError(f"positions [{pos}, {pos + n}) exceed a block table of "
                         f"{table.size} blocks")
    return table[k0:k1], pos - k0 * block_size


def _windows(spans, block_size: int) -> tuple:
    """The :func:`table_window` of each ``(table, pos, n)``: the windows concatenated, and
    per item ``(pos, offset)`` (``pos`` within its window, which starts at ``offset``)."""
    tabs, rows, off = [], [], 0
    for table, pos, n in spans:
        k0 = pos // block_size
        k1 = -(-(pos + n) // block_size)
        if pos < 0 or k1 > table.size:
            table_window(table, pos, n, block_size)  # raises
        tabs.append(table[k0:k1])
        rows.append((pos - k0 * block_size, off))
        off += k1 - k0
    return tabs[0] if len(tabs) == 1 else np.concatenate(tabs), rows


def paged_index(items: list, block_size: int):
    """Address the paged side of a batch of loads or saves: ``(mode, index, rows)``.

    When no item carries host slots, each item's window of its block table (the blocks
    its positions touch) is concatenated (int32) and the item gets ``(pos, offset)``:
    position ``pos + i`` resolves through ``table[offset + (pos + i) // block_size]`` on
    the device.  Otherwise the slots are concatenated (int64; ``from_blocks`` items are
    expanded on the host) and each item gets ``(0, offset)`` into them.
    """
    if all([it.slots is None for it in items]):
        spans = []
        tables: dict[int, np.ndarray] = {}  # items of one request share its block table
        for it in items:
            t = it.block_ids
            if type(t) is not np.ndarray or t.dtype != np.int32 or t.ndim != 1:
                ids = t
                t = tables.get(id(ids))
                if t is None:
                    t = tables[id(ids)] = _int32_table(ids)
            spans.append((t, int(it.dst_start), max(int(it.n_tokens), 0)))
        return ("table", *_windows(spans, block_size))
    parts, rows, off = [], [], 0
    for it in items:
        if it.slots is None:
            sl = host_slots(it.block_ids, it.paged_pos, it.paged_pos + it.n, block_size)
        else:
            sl = it.slots.to(torch.int64).reshape(-1)
        parts.append(sl)
        rows.append((0, off))
        off += int(sl.numel())
    return "slots", torch.cat(parts), rows


def detect_hnd(shape, block_size: int) -> bool:
    """HND ``[blocks, heads, bs, 2D]`` vs NHD ``[blocks, bs, heads, 2D]``; an ambiguous
    shape is NHD, vLLM's default (vllm_shift_connector.py:396-402)."""
    assert len(shape) == 4, f"expected fused 4-D KV layout, got {tuple(shape)}"
    hnd = shape[2] == block_size and shape[1] != block_size
    if shape[1] == block_size and shape[2] == block_size:
        hnd = False
    return hnd


def paged_planes(kv: torch.Tensor, block_size: int):
    """``(layout, k, v)`` of one layer's paged cache.

    4-D: the reference's fused cache (:396-402), rows ``[2D]``; ``k`` is the cache and
    ``v`` is None.  5-D: split K and V planes along the axis of size 2, as vLLM's
    ``[2, blocks, bs, heads, D]`` and ``[blocks, 2, bs, heads, D]`` caches hold them;
    ``k`` and ``v`` are the two planes (views), rows ``[D]``.  The layout of the 4-D
    cache or plane follows :func:`detect_hnd`.  A split cache of exactly two blocks has
    the same shape and strides in both forms; it is read as ``[2, blocks, ...]``,
    vLLM's default.
    """
    shape = tuple(kv.shape)
    if len(shape) == 4:
        return ("hnd" if detect_hnd(shape, block_size) else "nhd"), kv, None
    if len(shape) != 5 or 2 not in shape[:2]:
        raise ValueError(f"expected a fused 4-D or a split 5-D KV cache, got {shape}")
    axis = 0 if shape[0] == 2 else 1
    k, v = kv.select(axis, 0), kv.select(axis, 1)
    return ("hnd" if detect_hnd(tuple(k.shape), block_size) else "nhd"), k, v


def accept_multi(loads: list, num_computed: int, num_prompt_tokens: int, block_size: int,
                 covers) -> list:
    """Block-align every segment of a multi-segment load (vllm_shift_connector.py:225-245).

    ``covers(src_start, n)`` is the store's coverage check.  A segment is dropped, never
    guessed at, when alignment leaves less than a block, when it lies inside what the
    engine already holds, or when the store lost its source.
    """
    limit = (num_prompt_tokens - 1) // block_size * block_size
    floor = -(-num_computed // block_size) * block_size
    out = []
    for ld in loads:
        delta = int(ld["delta"])
        lo = max(-(-int(ld["dst_start"]) // block_size) * block_size, floor)
        hi = min(int(ld["dst_end"]), limit) // block_size * block_size
        if hi - lo < block_size:
            continue
        if not covers(lo - delta, hi - lo):
            continue
        out.append({"dst_start": lo, "dst_end": hi, "delta": delta})
    return out


class ShiftLoader:
    """Loads reused spans from a session store (the flat :class:`ShiftStore` or the
    :class:`BlockShiftStore`) into registered paged caches."""

    def __init__(
        self,
        store: ShiftStore | BlockShiftStore,
        block_size: int,
        inv_freq: torch.Tensor,
        *,
        k_scales: dict | None = None,
        timing: bool = False,
        verify: bool | None = None,
    ):
        self.store = store
        self.verify = VERIFY_LOAD if verify is None else bool(verify)
        self.verify_log: list = []  # one dict per (load, layer) checked
        self.block_size = int(block_size)
        self.inv_freq = inv_freq.detach().to(torch.float32).cpu()
        self.k_scales = k_scales if k_scales is not None else {}  # shared, may fill later
        self.timing = timing
        self._kv: dict[str, torch.Tensor] = {}
        self._planes: dict[str, tuple] = {}  # name -> (K, V or None), see paged_planes
        self.layout: str | None = None
        self.hnd: bool | None = None
        self.split = False
        self.head_size: int | None = None
        self.last_plan: ShiftPlan | SmallShifts | None = None
        self._sets = _CacheSets(self.block_size)
        self._small = _SmallRunners()
        self._k_scale_key: list | None = None
        self._k_scale_t: torch.Tensor | None = None

    @property
    def layer_names(self) -> list:
        """The registered layers, in the order their caches were given."""
        return list(self._kv)

    def register_kv_caches(self, kv_caches: dict) -> None:
        """Record the per-layer paged caches and their layout (:393-412): fused 4-D, as
        the reference takes them, or split K and V planes (5-D, :func:`paged_planes`)."""
        self._kv = dict(kv_caches)
        self._planes = {}
        for name, t in self._kv.items():
            layout, k, v = paged_planes(t, self.block_size)
            self._planes[name] = (k, v)
        self.layout = layout
        self.hnd = layout == "hnd"
        self.split = v is not None
        self.head_size = k.shape[3] if self.split else k.shape[3] // 2
        planes = list(self._planes.values())
        self._paged = CacheSet([[k for k, _ in planes]], layout, self.block_size,
                               v_caches=[[v for _, v in planes]] if self.split else None)
        one = next(iter(self._kv.values()))
        if one.is_cuda:
            _lib.lib()  # the kernels are compiled ahead of time: only load the library

    def start_load_kv(self, loads: list) -> int:
        """Issue every load of the step as one launch; returns token-layers loaded.

        Mirrors :481-534: each (load, layer) source is checked through the store (its
        ``read`` accounting: counters and LRU order move exactly as in the reference),
        and a load whose source is missing for any layer is logged and ends the step's
        loading.  Divergence: the reference has already written the layers before the
        missing one when it stops; here a missed load writes nothing.
        """
        if not loads or not self._kv:
            return 0
        names = list(self._kv)
        blocky = isinstance(self.store, BlockShiftStore)
        groups: dict[str, int] = {}
        taken = []
        for load in loads:
            n = load.n
            if n == 0:
                continue
            missing = self.store.lookup_layers(load.session, names, load.src_start, n)
            if missing is not None:
                logger.error(
                    "shift: session %s has no stored KV for %s; load skipped", load.session, missing
                )
                break
            groups.setdefault(load.session, len(groups))
            taken.append(load)
        if not taken:
            return 0
        dst_mode, dst_index, dst_rows = paged_index(taken, self.block_size)
        rows = []
        if blocky:
            # one pool per layer (K and V planes, or fused rows); each load's window of
            # its session's block table is the source index
            caches, v_caches = self.store.kernel_views(names)
            src = self._sets.get("store", [caches], "nhd", self.store.block_size,
                                 v_caches=None if v_caches is None else [v_caches])
            src_mode = "table"
            src_index, src_rows = _windows(
                [(self.store.table(ld.session), ld.src_start, ld.n) for ld in taken],
                self.store.block_size)
            for load, (spos, sidx), (dpos, didx) in zip(taken, src_rows, dst_rows):
                rows.append((spos, dpos, sidx, didx, load.n, int(load.delta), 0, 0))
        else:
            src = self._sets.get(
                "store", [[self.store.buffer(sess, name) for name in names] for sess in groups],
                "flat")
            src_mode, src_index = "flat", None
            for load, (dpos, didx) in zip(taken, dst_rows):
                rows.append((load.src_start, dpos, 0, didx, load.n, int(load.delta),
                             groups[load.session], 0))
        dst = self._paged
        k_scale = None
        if dst.first.dtype == torch.float8_e4m3fn:
            k_scale = self._k_scale(names)
        tokens = sum(load.n for load in taken)
        t0 = 0.0
        if self.timing:
            torch.cuda.synchronize(dst.first.device)
            t0 = time.perf_counter()
        # (slots on the GPU: a plan reads them there, in place)
        small = None if dst_mode == "slots" and dst_index.is_cuda else self._small.get(
            src, dst, src_mode, dst_mode, self.inv_freq, k_scale)
        if small is not None and small.fits(len(rows), tokens):  # no plan to build
            small.run(rows, _host(src_index), _host(dst_index), tokens=tokens)
            plan = small
        else:
            plan = ShiftPlan(
                np.array(rows, dtype=_lib.SPAN_DTYPE),
                src,
                dst,
                inv_freq=self.inv_freq,
                src_mode=src_mode,
                src_index=src_index,
                dst_mode=dst_mode,
                dst_index=dst_index,
                k_scale=k_scale,
                order="none",  # built for one launch: sorting would cost the step more
            )
            plan.launch()
        self.last_plan = plan
        if self.verify:
            for load in taken:
                for name in names:
                    self._verify(name, load, k_scale, names.index(name))
        if self.timing:
            torch.cuda.synchronize(dst.first.device)
            ms = (time.perf_counter() - t0) * 1e3
            logger.info(
                "shift: %d loads, %d tokens x %d layers, copy_ms=%.3f (%.1f GB/s)",
                len(rows),
                tokens,
                len(names),
                ms,
                plan.algorithmic_bytes / 1e9 / max(ms / 1e3, 1e-12),
            )
        return tokens * len(names)

    def _source_rows(self, load: Load, name: str) -> torch.Tensor:
        """``[n, heads, 2D]`` rows the load read, without the store's read accounting."""
        n = load.n
        if isinstance(self.store, BlockShiftStore):
            return self.store.gather(load.session, name, load.src_start, n)
        return self.store.buffer(load.session, name)[load.src_start:load.src_start + n]

    def _k_scale(self, names) -> torch.Tensor:
        """The layers' K scales as one fp32 CPU tensor, rebuilt only when a scale changed
        (``k_scales`` is shared with the saver and may fill in later)."""
        get = self.k_scales.get
        key = [float(get(name, 1.0)) for name in names]
        if self._k_scale_key != key:
            self._k_scale_key = key
            self._k_scale_t = torch.tensor(key, dtype=torch.float32)
        return self._k_scale_t

    def _verify(self, name: str, load: Load, k_scale, layer: int) -> None:
        """Read a loaded span back and compare it with torch's rotation of its source
        rows (vllm_shift_connector.py:444-480): K re-rotated by delta in fp32, the
        dimensions past ``rotary`` and V as stored.  fp8 rows are compared dequantised
        with the layer's K scale (V raw).  The figures are logged and kept in
        :attr:`verify_log`."""
        kp, vp = self._planes[name]
        row = self._source_rows(load, name)
        d = row.shape[-1] // 2
        rot = 2 * int(self.inv_freq.numel())
        slots = (load.slots if load.slots is not None else
                 host_slots(load.block_ids, load.paged_pos, load.paged_pos + load.n,
                            self.block_size)).to(kp.device, torch.int64)
        blk, off = slots // self.block_size, slots % self.block_size

        def rows_of(t):
            return t[blk, :, off] if self.hnd else t[blk, off]

        got = rows_of(kp) if vp is None else torch.cat((rows_of(kp), rows_of(vp)), dim=-1)
        scale = 1.0 if k_scale is None else float(k_scale[layer])
        k = row[..., :d].to(torch.float32) * scale
        want_k = torch.cat((_rerotate(k[..., :rot], int(load.delta), self.inv_freq),
                            k[..., rot:]), dim=-1)
        want = torch.cat((want_k, row[..., d:].to(torch.float32)), dim=-1)
        got = torch.cat((got[..., :d].to(torch.float32) * scale,
                         got[..., d:].to(torch.float32)), dim=-1)
        diff = (got - want).abs()
        entry = {
            "layer": name,
            "delta": int(load.delta),
            "n": int(load.n),
            "max_abs": float(diff.max()),
            "max_rel": float(diff.max() / want.abs().max().clamp_min(1e-6)),
            "mean_abs": float(diff.mean()),
            "v_exact": bool(torch.equal(got[..., d:], want[..., d:])),
        }
        self.verify_log.append(entry)
        logger.info("shift-verify: layer=%s delta=%d n=%d max_abs=%.4g max_rel=%.4g "
                    "mean_abs=%.4g", name, entry["delta"], entry["n"], entry["max_abs"],
                    entry["max_rel"], entry["mean_abs"])


@dataclass
class StepMeta:
    """What the scheduler hands the worker for one engine step: the step's loads, then
    its saves (the reference's ShiftConnectorMetadata, vllm_shift_connector.py:143-156)."""

    loads: list
    saves: list


class ShiftScheduler:
    """The connector's scheduler half over plain values (vllm_shift_connector.py:211-389).

    A request's ``kv_transfer_params`` (``{"session", "load": {dst_start, dst_end,
    delta}, "save": True | "full"}``, :16-18) come in; each engine step's
    :class:`StepMeta` goes out, for :class:`ShiftLoader` and :class:`ShiftSaver`.  The
    decisions are the reference's: one in-flight writer per session (:211-223);
    ``plan_load`` against the scheduler's store (:247-288); a load issued once, in the
    request's first scheduled step (:332-355); a save planned in every step, the
    one-shot ``"full"`` widening to ``[0, hi)`` then downgraded (:296-330).  ``store``
    is the scheduler's tensor-free mirror (``allocate=False``) of the worker's store:
    both reach the same decisions from the same calls.

    Loads and saves carry the request's block table (device-side slots,
    :meth:`Load.from_blocks`), or host slot lists with ``device_slots=False``, as the
    reference builds them.  The multi-segment ``"loads"`` path needs vLLM's gap-fill
    patch (:247-271) and is not wired here; :func:`accept_multi` is its alignment.
    """

    def __init__(self, store, block_size: int, *, device_slots: bool = True):
        from .shift_store import SessionTable

        self.store = store
        self.block_size = int(block_size)
        self.device_slots = bool(device_slots)
        self.table = SessionTable()
        self._params: dict[str, dict] = {}
        self._plans: dict[str, tuple] = {}
        self._blocks: dict[str, list] = {}
        self._need_load: set[str] = set()
        self._step_tables: dict[str, np.ndarray] = {}
        self._np_tables: dict[str, np.ndarray] = {}
        self.declines: list[str] = []

    def on_new_request(self, rid: str, params: dict | None) -> None:
        """Record the request's params; take the session's single writer slot."""
        params = dict(params or {})
        self._params[rid] = params
        session = params.get("session")
        if session and not self.table.acquire(rid, str(session)):
            logger.warning("shift: session %s already has an in-flight writer; request %s "
                           "runs with no reuse", session, rid)

    def get_num_new_matched_tokens(self, rid: str, num_computed: int,
                                   num_prompt_tokens: int) -> tuple[int, bool]:
        """Tokens the store will provide past the local prefix hit (``plan_load``)."""
        from .shift_store import plan_load

        session = self.table.session_of(rid)
        params = self._params.get(rid) or {}
        req = params.get("load")
        decision, why = plan_load(self.store, session, req, num_computed, num_prompt_tokens,
                                  self.block_size)
        if decision is None:
            if session and req:
                self.declines.append(why)
                logger.warning("shift: session %s declining reuse: %s", session, why)
            return 0, False
        self._plans[rid] = (decision.lo, decision.hi, decision.delta)
        return decision.hi - decision.lo, False

    def update_state_after_alloc(self, rid: str, num_external_tokens: int) -> None:
        if num_external_tokens > 0:
            self._need_load.add(rid)

    def _table_of(self, rid: str):
        """The request's block table as of this step (int32), one object per request per
        step: a step's load and saves of one request then share it.  Kept as a numpy
        array that grows with the request, so a decode step converts no list."""
        tab = self._step_tables.get(rid)
        if tab is None:
            blocks = self._blocks[rid]
            have = self._np_tables.get(rid)
            if have is None or have.size > len(blocks):
                have = np.asarray(blocks, np.int32)
            elif have.size < len(blocks):
                have = np.concatenate((have, np.asarray(blocks[have.size:], np.int32)))
            self._np_tables[rid] = have
            tab = self._step_tables[rid] = have
        return tab

    def _load(self, rid: str, lo: int, hi: int, delta: int) -> Load:
        session = self.table.session_of(rid) or ""
        if self.device_slots:
            return Load.from_blocks(session, self._table_of(rid), lo, hi, delta)
        return Load(session, host_slots(self._blocks[rid], lo, hi, self.block_size), lo - delta,
                    delta)

    def _plan_save(self, meta: StepMeta, rid: str, lo: int, hi: int) -> None:
        """Queue the save of the positions [lo, hi) this step computed, in the window
        ``plan_save`` grants (the reference's scheduler step,
        vllm_shift_connector.py:296-330).  A request that asked for a save and is
        refused one is logged with the reference's message.  ``"full"`` is one-shot: once
        a window has been granted, the request saves incrementally, so decode steps do
        not re-gather the whole prompt."""
        from .shift_store import plan_save

        if not self._blocks.get(rid):
            return  # no block table yet: nothing the kernels could read
        session = self.table.session_of(rid)
        params = self._params.get(rid, {})
        mode = params.get("save")
        window = plan_save(self.store, session, mode, lo, hi)
        if window is not None:
            if mode == "full":
                params["save"] = True
            meta.saves.append(self._save_item(rid, session or "", *window))
        elif mode and session and hi > lo:
            logger.warning("shift: session %s refused save of [%d,%d)", session, lo, hi)

    def _save_item(self, rid: str, session: str, lo: int, hi: int) -> Save:
        """A granted save window as the worker takes it: the request's block table
        (slots resolved on the device) or host slots."""
        if self.device_slots:
            return Save.from_blocks(session, self._table_of(rid), lo, hi)
        return Save(session, host_slots(self._blocks[rid], lo, hi, self.block_size), lo)

    def build_connector_meta(self, new_reqs=(), cached_reqs=(), finished=()) -> StepMeta:
        """One engine step.  ``new_reqs``: ``(rid, block_ids, num_computed_tokens,
        num_scheduled_tokens)`` of requests scheduled for the first time;
        ``cached_reqs``: ``(rid, new_block_ids or None, num_computed_tokens,
        num_scheduled_tokens)``; ``finished``: request ids to forget."""
        meta = StepMeta([], [])
        self._step_tables = {}
        for rid, block_ids, computed, scheduled in new_reqs:
            self._blocks[rid] = list(block_ids)
            self._np_tables.pop(rid, None)  # a request scheduled anew gets a new table
            if rid in self._need_load:
                lo, hi, delta = self._plans[rid]
                meta.loads.append(self._load(rid, lo, hi, delta))
                self._need_load.discard(rid)
            self._plan_save(meta, rid, computed, computed + scheduled)
        for rid, new_blocks, computed, scheduled in cached_reqs:
            if new_blocks is not None:
                self._blocks.setdefault(rid, []).extend(new_blocks)
            self._plan_save(meta, rid, computed, computed + scheduled)
        for rid in finished:
            self._forget(rid)
        return meta

    def request_finished(self, rid: str) -> None:
        """Forget the request and free its session's writer slot (:385-389)."""
        self._forget(rid)
        logger.info("shift: store %s", self.store.stats())

    def _forget(self, rid: str) -> None:
        self._blocks.pop(rid, None)
        self._np_tables.pop(rid, None)
        self._params.pop(rid, None)
        self._plans.pop(rid, None)
        self._need_load.discard(rid)
        self.table.release(rid)


class ShiftSaver:
    """Save path: paged cache -> session store, gathered on the device.

    The reference's ``save_kv_layer`` (vllm_shift_connector.py:539-553) reserves the
    span, gathers ``[T, heads, 2D]`` with advanced indexing (``_gather``, :418-442) and
    copies it into the store buffer (``ShiftStore.write``, shift_store.py:225-236).
    Here the gather kernel reads the paged rows and writes them straight into each
    session's buffer (delta 0: a pure copy), one launch for every save of the call.
    With a :class:`BlockShiftStore`, the rows land in the layer's pool through the
    session's block table, so a save never reallocates and never copies what is stored.
    """

    def __init__(self, store: ShiftStore | BlockShiftStore, block_size: int, *,
                 deferred: bool = False):
        self.store = store
        self.block_size = int(block_size)
        self.deferred = bool(deferred)
        self.last_plan: ShiftPlan | SmallShifts | None = None
        self._sets = _CacheSets(self.block_size)
        self._pending: list = []  # deferred: (layer name, paged cache, the step's saves)
        self.record = self._pending.append  # such a triple, for the next wait_for_save
        self._geo: dict[tuple, tuple] = {}  # the caches of a step -> their geometry
        self._small = _SmallRunners()

    def _geometry(self, caches: list) -> tuple:
        """``(row_shape, dtype, device, paged CacheSet, caches)`` of a step's paged caches,
        worked out once per distinct tuple of cache tensors (vLLM passes the same ones every
        step)."""
        # keyed by the tensors' ids (a tuple of tensors would hash each tensor through
        # Python); the entry holds the tensors, so no id is reused meanwhile (its CacheSet
        # alone does not: of split caches it has views, which need not keep their base)
        key = tuple(map(id, caches))
        hit = self._geo.get(key)
        if hit is None:
            planes = [paged_planes(t, self.block_size) for t in caches]
            layout, first, v_first = planes[0]
            split = v_first is not None
            # the store holds fused rows [heads, 2D] whichever way the cache keeps them
            row_shape = (first.shape[1] if layout == "hnd" else first.shape[2],
                         first.shape[3] * (2 if split else 1))
            paged = CacheSet([[k for _, k, _ in planes]], layout, self.block_size,
                             v_caches=[[v for _, _, v in planes]] if split else None)
            if len(self._geo) >= 64:  # caches replaced many times over
                self._geo.clear()
            hit = self._geo[key] = (row_shape, first.dtype, first.device, paged, tuple(caches))
        return hit

    def _plan(self, names: list, caches: list, saves: list) -> int:
        row_shape, dtype, device, paged, _ = self._geometry(caches)
        if isinstance(self.store, BlockShiftStore):
            return self._plan_blocks(names, saves, row_shape, dtype, device, paged)
        groups: dict[str, int] = {}
        bufs: list[list] = []
        taken = []
        for save in saves:
            n = save.n
            if n == 0:
                continue
            # mirrors the scheduler's reserve for this step; idempotent across layers
            if not self.store.reserve(save.session, save.dst_start, n):
                continue
            targets = self.store.write_targets(save.session, names, save.dst_start, n,
                                               row_shape, dtype, device)
            if targets is None:
                continue
            g = groups.get(save.session)
            if g is None:
                g = groups[save.session] = len(bufs)
                bufs.append(targets)
            else:
                bufs[g] = targets  # a save may have grown (reallocated) the buffers
            taken.append(save)
        if not taken:
            return 0
        src_mode, src_index, src_rows = paged_index(taken, self.block_size)
        rows = []
        dst = self._sets.get("store", bufs, "flat")
        for sv, (spos, sidx) in zip(taken, src_rows):
            rows.append((spos, int(sv.dst_start), sidx, 0, sv.n, 0, 0, groups[sv.session]))
        return self._launch(names, paged, dst, rows, src_mode, src_index, "flat", None)

    def _plan_blocks(self, names: list, saves: list, row_shape, dtype, device, paged) -> int:
        store = self.store
        taken = store.take_saves(saves, names, row_shape, dtype, device)
        if not taken:
            return 0
        caches, v_caches = store.kernel_views(names)
        dst = self._sets.get("store", [caches], "nhd", store.block_size,
                             v_caches=None if v_caches is None else [v_caches])
        src_mode, src_index, src_rows = paged_index([t[0] for t in taken], self.block_size)
        dst_index, dst_rows = _windows(
            [(entry.table, sv.dst_start, n) for sv, entry, n in taken], store.block_size)
        rows = [(spos, dpos, sidx, didx, n, 0, 0, 0)
                for (_, _, n), (spos, sidx), (dpos, didx) in zip(taken, src_rows, dst_rows)]
        return self._launch(names, paged, dst, rows, src_mode, src_index, "table", dst_index)

    def _launch(self, names: list, paged, dst, rows: list, src_mode, src_index, dst_mode,
                dst_index) -> int:
        tokens = sum([r[4] for r in rows])
        # (slots on the GPU: a plan reads them there, in place)
        small = None if src_mode == "slots" and src_index.is_cuda else self._small.get(
            paged, dst, src_mode, dst_mode, None)
        if small is not None and small.fits(len(rows), tokens):  # no plan to build
            small.run(rows, _host(src_index), _host(dst_index), tokens=tokens)
            self.last_plan = small
            return tokens * len(names)
        plan = ShiftPlan(
            np.array(rows, dtype=_lib.SPAN_DTYPE),
            paged,
            dst,
            inv_freq=None,
            src_mode=src_mode,
            src_index=src_index,
            dst_mode=dst_mode,
            dst_index=dst_index,
            order="none",  # built for one launch: sorting would cost the step more
        )
        plan.launch()
        self.last_plan = plan
        return tokens * len(names)

    def save_kv_layer(self, layer_name: str, kv_layer: torch.Tensor, saves: list) -> int:
        """One layer, every save of the step (the reference's per-layer hook).

        Deferred (``deferred=True``): the layer is only recorded, and returns 0; the
        step's :meth:`wait_for_save` saves every recorded layer in one launch.  vLLM
        calls that hook at the end of the forward pass, when every layer's KV for the
        step is final, and the store ends the step in the state per-layer saves leave.
        """
        if self.deferred:
            self.record((layer_name, kv_layer, saves))
            return 0
        return self._plan([layer_name], [kv_layer], saves)

    def wait_for_save(self) -> int:
        """Flush the deferred layers: one launch per distinct list of saves (a step has
        one).  Returns the token-layers saved; 0 when nothing is pending."""
        pending = self._pending[:]
        del self._pending[:len(pending)]  # not what another thread has recorded since
        if not pending:
            return 0
        saves = pending[0][2]
        if all([item[2] is saves for item in pending]):
            names, caches, _ = zip(*pending)
            return self._plan(names, caches, saves)
        groups: dict[int, tuple] = {}
        for name, cache, saves in pending:
            names, caches, _ = groups.setdefault(id(saves), ([], [], saves))
            names.append(name)
            caches.append(cache)
        return sum(self._plan(names, caches, saves) for names, caches, saves in groups.values())

    def save_all(self, kv_caches: dict, saves: list) -> int:
        """Every layer and every save of the step in one launch (at the end of a step)."""
        names = list(kv_caches)
        return self._plan(names, [kv_caches[n] for n in names], saves)
