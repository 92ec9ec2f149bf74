"""The cache on the device.

Keys and values live in pages of 64 tokens. Layers are partitioned into groups
by what they keep (kv heads, key and value widths, all keys or a window of them); each
group has pools of its own, [runs][pages][kv_heads][elements of a page] for K and for
V, a page as large as the group's mixers ask for (KVNeed.k_elems, KVNeed.v_elems: the order
inside a page is theirs), and one page table [slots][blocks]
shared by its runs. A sequence holds a
slot: its row of every page table, its length, and its row of the fixed-size
state area. Slots and pages go back to the free lists when a sequence ends and
are handed out again, lowest first; nothing is cleared, because attention only
reads positions a sequence has written (the reference argues the same for its
rewind: src/kv_cache.hpp:93-96). The reference's cache is one
[layers][batch][max_seq][kv_heads][head_dim] block with a single position
(src/kv_cache.hpp:161-203); slots, pages and groups are this engine's own.
"""
from __future__ import annotations

import dataclasses

import numpy as np
import torch

from ..kernels import ops
from ..parts.base import KVNeed, LayerCache
from .pages import PAGE_TOKENS, CacheError, CacheFull, GroupPages, SlotBook, blocks_for  # noqa: F401


@dataclasses.dataclass
class RunPlan:
    """What one run of the schedule needs from the cache."""

    kv: KVNeed | None          # keys/values it writes (None: none, or it reads another run's)
    cache_from: int | None     # run whose keys/values it reads
    state_bytes: int = 0


class _Group:
    def __init__(self, need: KVNeed, runs: list[int], num_pages: int, dtype, device, tables: "_Tables", index: int):
        self.need = need
        self.runs = runs
        # zero-filled once (as the reference's cache is: src/kv_cache.hpp:161-203): a masked
        # key still enters the matrix products with weight 0, so it must never be NaN
        # a page is as large as the mixers of the group say; what lies where inside it is theirs
        self.kpool = torch.zeros((len(runs), num_pages, need.kv_heads, need.k_elems), dtype=dtype, device=device)
        self.vpool = torch.zeros((len(runs), num_pages, need.kv_heads, need.v_elems), dtype=dtype, device=device)
        self._tables = tables
        self._table = tables.device[index]
        # the same table on the host: a step can take its sequences' rows along with its metadata
        self.host_table = tables.host[index]

    @property
    def page_table(self) -> torch.Tensor:
        self._tables.flush()
        return self._table


class _Tables:
    """The groups' page tables [groups][slots][blocks], on the host and on the device. Entries change on the host at once and
    on the device all together before the next step (flush): one copy from pinned memory and one launch behind what is
    queued. (Written slot by slot, from pageable memory, every release, truncation and new page made the host wait for
    all queued steps and left the GPU idle for 60 us behind them: 64 sequences cut back after eight steps, 21 of them by a
    page, 1.3 ms of 17.2.) The pinned memory is there from the start: TURNS parts of TURN entries, used in turn, each free again when its
    event has passed; more entries than a part holds go in several launches. (Made by the steps that first wanted it, each of the
    first four and every one with more entries than before had a host allocation in its path.)"""

    TURNS, TURN = 4, 4096

    def __init__(self, groups: int, max_slots: int, max_blocks: int, device):
        self.host = np.full((groups, max_slots, max_blocks), -1, dtype=np.int32)
        self.device = torch.full((groups, max_slots, max_blocks), -1, dtype=torch.int32, device=device)
        self._flat = self.host.reshape(-1)
        self._dirty: set[int] = set()
        self._turn = max(1, min(self.TURN, self._flat.size))
        self._pinned: list[torch.Tensor] = []
        if self.device.device.type != "cpu":
            self._pinned = list(torch.empty((self.TURNS, 2 * self._turn), dtype=torch.int32, pin_memory=True))
        self._events: list[torch.cuda.Event | None] = [None] * self.TURNS
        self._next = 0

    def write(self, index: int, page: int) -> None:
        self._flat[index] = page
        self._dirty.add(index)

    def flush(self) -> None:
        n = len(self._dirty)
        if n == 0:
            return
        idx = np.fromiter(self._dirty, dtype=np.int32, count=n)
        if self.device.device.type == "cpu":
            self.device.view(-1)[torch.from_numpy(idx).long()] = torch.from_numpy(self._flat[idx])
            self._dirty.clear()
            return
        for at in range(0, n, self._turn):
            self._send(idx[at:at + self._turn])
        self._dirty.clear()              # (only now: entries that an error kept from the device go with the next flush)

    def _send(self, idx: np.ndarray) -> None:
        i, n = self._next, len(idx)
        self._next = (i + 1) % self.TURNS
        if self._events[i] is not None:
            self._events[i].synchronize()
        staged = self._pinned[i][:2 * n]
        staged.numpy()[:n] = idx
        staged.numpy()[n:] = self._flat[idx]
        entries = torch.empty(2 * n, dtype=torch.int32, device=self.device.device)
        entries.copy_(staged, non_blocking=True)
        self._events[i] = torch.cuda.Event()
        self._events[i].record()
        ops.scatter_i32(self.device, entries, n)


class PagedCache:
    def __init__(self, plans: list[RunPlan], *, max_tokens: int, max_slots: int,
                 max_seq_len: int, dtype: torch.dtype, device):
        if max_tokens < PAGE_TOKENS:
            raise CacheError(f"max_tokens {max_tokens} is below one page of {PAGE_TOKENS} tokens")
        self.device = device
        self.dtype = dtype
        self.num_pages = max_tokens // PAGE_TOKENS
        self.max_slots = max(1, min(max_slots, self.num_pages))
        self.max_blocks = max(1, min(blocks_for(max_seq_len), self.num_pages))
        self.max_seq_len = self.max_blocks * PAGE_TOKENS
        self.plans = plans

        # group runs by what they keep
        keys: list[KVNeed] = []
        members: list[list[int]] = []
        self.run_group: dict[int, tuple[int, int]] = {}
        for r, plan in enumerate(plans):
            if plan.kv is None:
                continue
            if plan.kv not in keys:
                keys.append(plan.kv)
                members.append([])
            gi = keys.index(plan.kv)
            self.run_group[r] = (gi, len(members[gi]))
            members[gi].append(r)
        for r, plan in enumerate(plans):
            if plan.cache_from is not None:
                if plan.cache_from not in self.run_group or plan.cache_from >= r:
                    raise CacheError(f"run {r} reads the cache of run {plan.cache_from}, "
                                     "which is not an earlier run with a cache of its own")
        self.tables = _Tables(len(keys), self.max_slots, self.max_blocks, device)
        self.groups = [_Group(k, m, self.num_pages, dtype, device, self.tables, i) for i, (k, m) in enumerate(zip(keys, members))]
        self.book = SlotBook(self.max_slots, self.max_blocks,
                             [GroupPages(self.num_pages, k.window, f"{i}", k.chunk) for i, k in enumerate(keys)])

        # fixed-size per-sequence state: one row per slot, one span per run
        self.state_offsets: list[int] = []
        off = 0
        for plan in plans:
            self.state_offsets.append(off)
            off += (plan.state_bytes + 255) // 256 * 256
        self.state_bytes_per_slot = off
        self.state = torch.zeros((self.max_slots, off), dtype=torch.uint8, device=device) if off else None

    # -- slots --------------------------------------------------------------
    def acquire(self) -> int:
        slot = self.book.acquire()
        if self.state is not None:
            self.state[slot].zero_()
        return slot

    def release(self, slot: int) -> None:
        self._clear(self.book.release(slot))

    def truncate(self, slot: int, new_length: int) -> None:
        """Keeps the first new_length tokens of the slot and gives back the pages beyond
        (cache/pages.py: SlotBook.truncate). A model that keeps fixed-size state per
        sequence cannot be rewound: the state has seen the dropped tokens."""
        if self.state is not None and new_length < self.length(slot):
            raise CacheError(f"slot {slot}: a model with per-sequence state cannot be truncated")
        self._clear(self.book.truncate(slot, new_length))

    def length(self, slot: int) -> int:
        try:
            return self.book.length[slot]
        except KeyError:
            raise CacheError(f"slot {slot} is not held") from None

    @property
    def free_pages(self) -> int:
        return min((g.pool.available for g in self.book.groups), default=self.num_pages)

    # -- pages --------------------------------------------------------------
    def reserve(self, growth: list[tuple[int, int]]) -> None:
        """growth: (slot, new length) for every sequence of a step. Either all get
        their pages or none does."""
        for s, n in growth:            # every check before any page is taken
            if blocks_for(n) > self.max_blocks:
                raise CacheFull(f"slot {s}: {n} tokens exceed the longest sequence the cache was "
                                f"built for ({self.max_seq_len})")
        need = sum(self.book.pages_needed(s, n) for s, n in growth)
        for g in self.book.groups:
            if need > g.pool.available:
                raise CacheFull(f"the step needs {need} more pages of {PAGE_TOKENS} tokens per "
                                f"group, {g.pool.available} are free")
        if need == 0:       # most one-token steps: every new position already has its page
            for s, n in growth:
                if n < self.book.length[s]:
                    raise CacheError(f"slot {s}: cannot shrink from {self.book.length[s]} to {n}")
        else:
            added = []
            for s, n in growth:
                added += self.book.reserve(s, n)
            self._write(added)
        self.tables.flush()

    def commit(self, growth: list[tuple[int, int]]) -> None:
        cleared = []
        for s, n in growth:
            cleared += self.book.commit(s, n)
        self._clear(cleared)

    def _write(self, entries) -> None:
        for gi, slot, block, page in entries:
            self.tables.write((gi * self.max_slots + slot) * self.max_blocks + block, page)

    def _clear(self, entries) -> None:
        self._write([(gi, slot, block, -1) for gi, slot, block in entries])

    def rows_of_tables(self, slots: list[int], out: np.ndarray) -> None:
        """out[g, r, :] = the page table row of slots[r] in group g (int32 [groups, rows or more,
        max_blocks]; rows beyond the slots keep what they hold)."""
        for gi, g in enumerate(self.groups):
            out[gi, :len(slots)] = g.host_table[slots]

    # -- views for the layers -----------------------------------------------
    def layer_cache(self, run: int) -> LayerCache:
        plan = self.plans[run]
        src = run if plan.kv is not None else plan.cache_from
        state = None
        if plan.state_bytes:
            o = self.state_offsets[run]
            state = self.state[:, o:o + plan.state_bytes]
        if src is None:
            return LayerCache(None, None, None, False, state)
        gi, pi = self.run_group[src]
        g = self.groups[gi]
        return LayerCache(g.kpool[pi], g.vpool[pi], g.page_table, plan.kv is not None, state)

    def bytes_per_token(self) -> int:
        es = torch.empty((), dtype=self.dtype).element_size()
        return sum(len(g.runs) * g.need.kv_heads * es * (g.need.k_elems + g.need.v_elems) // PAGE_TOKENS
                   for g in self.groups)
