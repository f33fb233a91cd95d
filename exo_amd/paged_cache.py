"""Paged KV pool: pages of 64 positions shared by all sequences of a batch.

The cache protocol of ``ShardKVCache`` (rows, ``offsets``, ``pos``, trim / reset / copy_row) over a
pool whose size is given in tokens, not rows x longest sequence: a row owns the pages its tokens
need, through a page table on the device, and gives them back when it is trimmed, reset or
released.  One table serves every layer.  Recurrent layers keep their fixed-size states in slots beside
the pages (``state_pool``); a row then cannot be cut back to an earlier position, only to none.

Per layer with keys of its own (layers that use another layer's keys have no storage):
  k[i]  [pages, G, 64, ldk]   keys as attention uses them (normalised)
  v[i]  [pages, G, ldv, 64]   values, transposed inside the page (matrix-core operand order)
A layer whose queries see means over blocks of P positions keeps those too, in pages of 64 blocks laid out the
same way (``mean_k[i]``, ``mean_v[i]``), behind a table per block size: a block's mean is formed when its last
position is appended, and depends on nothing but the cached keys and values.
with ldk, ldv the head sizes rounded up to 32; the padding stays zero.  Latent attention keeps one "key" per
position - the normed latent, and behind it the shared rotated key part - and no values.
"""

from __future__ import annotations

import torch

from . import ops
from .cache import HostWrites, LayerKV
from .state_pool import StatePool, StateShape

PAGE = 64


class PoolExhausted(RuntimeError):
    """No free page for a token that is about to be appended."""


def pages_for(tokens: int) -> int:
    return -(-tokens // PAGE)


class PageTable:
    """Which pages hold a row's sequence, ``span`` positions each: lists here, a table on the device."""

    def __init__(self, rows: int, n_pages: int, span: int, max_pages: int, device):
        self.n_pages, self.span = n_pages, span
        self.table = torch.zeros(rows, max(1, max_pages), dtype=torch.int32, device=device)
        self.pages: list[list[int]] = [[] for _ in range(rows)]
        self.free = list(range(n_pages - 1, -1, -1))

    def missing(self, row: int, positions: int) -> int:
        return max(0, -(-positions // self.span) - len(self.pages[row]))

    def take(self, row: int, k: int) -> None:
        if k:
            new = [self.free.pop() for _ in range(k)]
            at = len(self.pages[row])
            self.pages[row] += new
            ops.put_ints(self.table[row, at : at + k], new)

    def give_back(self, row: int, keep: int) -> None:
        """All pages but those of the first ``keep`` positions."""
        n = -(-keep // self.span)
        self.free += reversed(self.pages[row][n:])
        del self.pages[row][n:]

    def move(self, src: int, dst: int) -> None:
        self.give_back(dst, 0)
        self.pages[dst], self.pages[src] = self.pages[src], []
        self.table[dst].copy_(self.table[src])

    def swap(self, a: int, b: int) -> None:
        self.pages[a], self.pages[b] = self.pages[b], self.pages[a]
        self.table[[a, b]] = self.table[[b, a]]


class PagedKVCache(HostWrites, list):
    """list[LayerKV] (one per layer with keys of its own and per recurrent state) plus the pools."""

    def __init__(self, layers: list[tuple[int, int, int]], rows: int, max_seq: int, device, dtype=torch.bfloat16,
                 pool_tokens: int | None = None, states: list[StateShape] = (), blocks: list[int | None] | None = None):
        """``layers``: (kv heads, key size, value size) per storing layer.  ``max_seq``: the longest
        sequence a row may hold; ``pool_tokens``: tokens all rows hold together, each row's count
        rounded up to whole pages (default: every row at ``max_seq``); ``states``: of the layers that keep
        one; ``blocks``: per storing layer the positions of a block whose means it keeps (None: it keeps none)."""
        super().__init__(LayerKV(self, i) for i in range(len(layers) + len(states)))
        self.batch, self.max_seq, self.shapes = rows, max_seq, list(layers)
        self.n_pages = rows * pages_for(max_seq) if pool_tokens is None else pages_for(pool_tokens)
        self.max_pages = min(pages_for(max_seq), self.n_pages)
        pad = lambda d: -(-d // 32) * 32  # noqa: E731
        z = dict(dtype=dtype, device=device)
        self.k = [torch.zeros(self.n_pages, g, PAGE, pad(d), **z) for g, d, _ in layers]
        self.v = [torch.zeros(self.n_pages, g, pad(e), PAGE, **z) for g, _, e in layers]
        self.states = StatePool(states, rows, device, dtype)
        self._main = PageTable(rows, self.n_pages, PAGE, self.max_pages, device)
        self.table, self.pages, self._free = self._main.table, self._main.pages, self._main.free
        # a row's whole blocks fill at most its own pages / P pages and part of one more: never short of pages
        # while the main pool has any
        self.blocks = [None] * len(layers) if blocks is None else list(blocks)
        self.means = {p: PageTable(rows, self.n_pages // p + rows, PAGE * p, self.max_pages // p + 1, device)
                      for p in sorted({p for p in self.blocks if p})}
        self.mean_k = [torch.zeros(self.means[p].n_pages, g, PAGE, pad(d), **z) if p else None
                       for (g, d, _), p in zip(layers, self.blocks)]
        self.mean_v = [torch.zeros(self.means[p].n_pages, g, pad(e), PAGE, **z) if p else None
                       for (g, _, e), p in zip(layers, self.blocks)]
        self.pos = torch.zeros(rows, dtype=torch.int32, device=device)
        self.offsets = [0] * rows
        self._last_trim = 0

    # -- recurrent states
    @property
    def trimmable(self) -> bool:
        """Whether a row can go back to an earlier position (a recurrent state cannot)."""
        return not len(self.states)

    def save_states(self, rows) -> list[torch.Tensor]:
        self.order()
        return self.states.read(rows)

    def load_states(self, rows, saved: list[torch.Tensor]) -> None:
        self.order()
        self.states.write(rows, saved)

    # -- pages
    @property
    def free_tokens(self) -> int:
        return len(self._free) * PAGE

    def reserve(self, rows, n: int) -> None:
        """Pages for ``n`` more tokens in each of ``rows``; raises before anything changes if a row
        or the pool cannot hold them."""
        self.reserve_each([(r, n) for r in rows])

    def reserve_each(self, wants: list[tuple[int, int]]) -> None:
        need = []
        for r, n in wants:
            if self.offsets[r] + n > self.max_seq:
                raise ValueError(f"KV cache overflow: {self.offsets[r]}+{n} > {self.max_seq}")
            need.append(self._main.missing(r, self.offsets[r] + n))
        if sum(need) > len(self._free):
            raise PoolExhausted(f"{sum(need)} pages of {PAGE} tokens wanted, {len(self._free)} free")
        self.order()
        taken = sum(need)
        for (r, n), k in zip(wants, need):
            self._main.take(r, k)
            for p, t in self.means.items():
                k = t.missing(r, self._whole(r, n, p))
                t.take(r, k)
                taken += k
        if taken:
            self._changed()

    def _whole(self, row: int, n: int, block: int) -> int:
        """Positions in whole blocks after ``n`` more tokens."""
        return (self.offsets[row] + n) // block * block

    def _give_back(self, row: int, keep_tokens: int) -> None:
        self._main.give_back(row, keep_tokens)
        for p, t in self.means.items():
            t.give_back(row, keep_tokens // p * p)

    # -- fill level (ShardKVCache's protocol)
    def advance_host(self, t: int, rows=None) -> None:
        for r in (range(self.batch) if rows is None else rows):
            self.offsets[r] += t

    def trim(self, n: int, rows=None) -> int:
        rows = range(self.batch) if rows is None else rows
        n = min([n] + [self.offsets[r] for r in rows])
        if n and not self.trimmable and any(self.offsets[r] != n for r in rows):
            raise ValueError("a recurrent state cannot be cut back to an earlier position")
        for r in rows:
            self.offsets[r] -= n
            self._give_back(r, self.offsets[r])
        self.sync_pos()
        return n

    def reset(self, rows=None) -> None:
        for r in (range(self.batch) if rows is None else rows):
            self.offsets[r] = 0
            self._give_back(r, 0)
        self.sync_pos()

    def release(self, row: int) -> None:
        """The row's sequence is finished: its pages go back to the pool."""
        self.reset(rows=[row])

    def copy_row(self, src: int, dst: int) -> None:
        """Move one sequence to another row (slot compaction): pages and state slot change hands,
        no key or state moves."""
        self.order()
        for t in (self._main, *self.means.values()):
            t.move(src, dst)
        self.offsets[dst], self.offsets[src] = self.offsets[src], 0
        self.states.swap(src, dst)
        self.sync_pos()

    def swap_rows(self, a: int, b: int) -> None:
        if a == b:
            return
        self.order()
        for t in (self._main, *self.means.values()):
            t.swap(a, b)
        self.offsets[a], self.offsets[b] = self.offsets[b], self.offsets[a]
        self.states.swap(a, b)
        self.sync_pos()

    def nbytes(self) -> int:
        return sum(t.numel() * t.element_size() for t in self.k + self.v + self.mean_k + self.mean_v if t is not None) + self.states.nbytes()

    # -- one row's contents as [n, G, size] tensors (prefix cache, wire)
    def _row_pages(self, row: int, lo: int, hi: int) -> torch.Tensor:
        return torch.tensor(self.pages[row][lo // PAGE : pages_for(hi)], dtype=torch.int64, device=self.pos.device)

    def read_nhd(self, layer: int, row: int, start: int, n: int) -> tuple[torch.Tensor, torch.Tensor]:
        """Keys [n, G, D] and values [n, G, E] of positions [start, start + n)."""
        self.order()
        g, d, e = self.shapes[layer]
        idx, off = self._row_pages(row, start, start + n), start % PAGE
        rows = len(idx) * PAGE
        k = self.k[layer][idx].permute(0, 2, 1, 3).reshape(rows, g, self.k[layer].shape[-1])
        v = self.v[layer][idx].permute(0, 3, 1, 2).reshape(rows, g, self.v[layer].shape[2])
        return k[off : off + n, :, :d].contiguous(), v[off : off + n, :, :e].contiguous()

    def write_nhd(self, layer: int, row: int, start: int, k: torch.Tensor, v: torch.Tensor) -> None:
        """Positions [start, start + n) from keys [n, G, D] and values [n, G, E]; the row must own
        their pages (``reserve``)."""
        n = k.shape[0]
        g, d, e = self.shapes[layer]
        if tuple(k.shape[1:]) != (g, d) or tuple(v.shape) != (n, g, e):
            raise ValueError(f"keys {tuple(k.shape)} / values {tuple(v.shape)} do not fit layer {layer} ({g}, {d}, {e})")
        self.order()
        at = torch.arange(start, start + n, device=self.pos.device)
        page = self._row_pages(row, 0, start + n)[at // PAGE]
        self.k[layer][page, :, at % PAGE, :d] = k.to(self.k[layer].dtype)
        self.v[layer][page, :, :e, at % PAGE] = v.to(self.v[layer].dtype)
        if self.blocks[layer]:
            self._write_means(layer, row, start, start + n)

    def _write_means(self, layer: int, row: int, start: int, end: int) -> None:
        """Means of the blocks whose last position lies in [start, end); all earlier positions are written."""
        p, (g, d, e) = self.blocks[layer], self.shapes[layer]
        lo, hi, t = start // p, end // p, self.means[self.blocks[layer]]
        if hi <= lo:
            return
        if missing := t.missing(row, hi * p):
            self.order()
            t.take(row, missing)
            self._changed()
        k, v = (x.float().view(hi - lo, p, *x.shape[1:]).mean(1) for x in self.read_nhd(layer, row, lo * p, (hi - lo) * p))
        at = torch.arange(lo, hi, device=self.pos.device)
        page = torch.tensor(t.pages[row], dtype=torch.int64, device=self.pos.device)[at // PAGE]
        self.mean_k[layer][page, :, at % PAGE, :d] = k.to(self.k[layer].dtype)
        self.mean_v[layer][page, :, :e, at % PAGE] = v.to(self.v[layer].dtype)

    def snapshot(self, row: int) -> list[tuple[torch.Tensor, torch.Tensor]]:
        """Detached copy of the row's positions, per layer (keys, values), then the recurrent
        states (one entry of all of them, if there are any)."""
        self.order()
        kv = [self.read_nhd(i, row, 0, self.offsets[row]) for i in range(len(self.k))]
        return kv + ([tuple(self.states.read([row]))] if len(self.states) else [])

    def restore(self, row: int, layers: list[tuple[torch.Tensor, torch.Tensor]], length: int) -> None:
        self.reset(rows=[row])
        self.reserve([row], length)
        if len(self.states):
            self.states.write([row], list(layers[-1]))
        for i, (k, v) in enumerate(layers[: len(self.k)]):
            self.write_nhd(i, row, 0, k[:length], v[:length])
        self.offsets[row] = length
        self.sync_pos()
