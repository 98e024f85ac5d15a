"""A step's saves taken together (``BlockShiftStore.take_saves``) against one
``reserve`` and ``write_targets`` per save: the same saves taken, block tables, windows,
counters, LRU order and layers, over random steps that append inside a block, open new
blocks, truncate, leave holes, repeat a session and evict others."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from marathon_amd.block_store import BlockShiftStore
from marathon_amd.connector import Save, ShiftSaver

ROW, DT = (2, 32), torch.bfloat16


def _one_by_one(store, saves, layers):
    taken = []
    for sv in saves:
        if sv.n == 0 or not store.reserve(sv.session, sv.dst_start, sv.n):
            continue
        if store.write_targets(sv.session, layers, sv.dst_start, sv.n, ROW, DT, "cpu") is None:
            continue
        taken.append(sv)
    if len(taken) > 1:
        taken = [sv for sv in taken if store.holds_blocks(sv.session, sv.dst_start, sv.n)]
    return taken


def _state(store):
    return [(s, e.base, e.filled, e.held, list(e.valid), e.table.tolist(), sorted(e.layers))
            for s, e in store._sessions.items()]


@pytest.mark.parametrize("allocate,truncate", [(True, True), (True, False), (False, True)])
@pytest.mark.parametrize("budget", [4096, 320])  # room for all; evictions
def test_take_saves_matches_one_by_one(budget, allocate, truncate):
    for seed in range(6):
        rng = np.random.default_rng(seed)
        a, b = (BlockShiftStore(budget, "cpu", allocate, 16, truncate) for _ in range(2))
        top = {f"s{k}": 0 for k in range(8)}
        for step in range(60):
            layers = ["l0", "l1", "l2"][:int(rng.integers(1, 4))]
            saves = []
            for s in rng.permutation(list(top))[:int(rng.integers(1, 9))]:
                at = int(rng.choice([top[s], top[s], top[s], max(0, top[s] - 20), top[s] + 3]))
                n = int(rng.choice([1, 1, 1, 0, 15, 40]))
                saves.append(Save.from_blocks(str(s), np.zeros(1, np.int32), at, at + n))
                top[s] = at + n if n else top[s]
            if rng.random() < 0.3:  # a session twice in one step
                saves.append(saves[0])
            got = a.take_saves(saves, layers, ROW, DT, "cpu")
            want = _one_by_one(b, saves, layers)
            assert [id(t[0]) for t in got] == [id(sv) for sv in want]
            assert all(t[1] is a._sessions[t[0].session] and t[2] == t[0].n for t in got)
            assert _state(a) == _state(b)
            assert a.stats() == b.stats() and sorted(a._free) == sorted(b._free)
            top = {s: a._sessions[s].filled if s in a._sessions and truncate else top[s]
                   for s in top}
            assert list(a._pools) == list(b._pools)


def test_deferred_layers_are_grouped_by_their_saves():
    """``wait_for_save`` plans one batch per distinct list of saves, in the order the
    lists first appear, however the layers' calls interleave."""
    saver = ShiftSaver(BlockShiftStore(64, "cpu"), 16, deferred=True)
    seen = []
    saver._plan = lambda names, caches, saves: seen.append((list(names), list(caches), saves)) or 1
    one, two = [1], [1]
    for name, saves in (("a", one), ("b", one), ("c", two), ("d", one)):
        assert saver.save_kv_layer(name, name.upper(), saves) == 0
    assert saver.wait_for_save() == 2
    assert seen == [(["a", "b", "d"], ["A", "B", "D"], one), (["c"], ["C"], two)]
    assert seen[0][2] is one and seen[1][2] is two
    saver.save_kv_layer("e", "E", two)
    assert saver.wait_for_save() == 1 and seen[2] == (["e"], ["E"], two)
    assert saver.wait_for_save() == 0


def test_a_layer_recorded_while_the_step_is_flushed_is_kept():
    """A hook on another thread between the flush's copy and its clearing of the list."""
    saver = ShiftSaver(BlockShiftStore(64, "cpu"), 16, deferred=True)
    one, two, seen = [1], [1], []

    class Pending(list):
        def __getitem__(self, key):
            got = super().__getitem__(key)
            if self:
                self.append(("late", "LATE", two))
            return got

    saver._pending = Pending([("a", "A", one)])
    saver._plan = lambda names, caches, saves: seen.append((list(names), saves)) or 1
    assert saver.wait_for_save() == 1
    saver._pending = list(saver._pending)
    assert saver.wait_for_save() == 1
    assert seen == [(["a"], one), (["late"], two)] and seen[1][1] is two
