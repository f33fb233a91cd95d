"""The forward of layer-list decoders (``stack_config``) over a paged KV pool.

One step function serves everything: ``step(cache, entries)`` takes, per sequence, the cache row
and its next tokens - a portion of a prompt, a single decoded token, or both kinds side by side in
one batch - runs them together and returns logits at the places asked for.  ``__call__`` and
``decode_step`` (the graph-captured single-token step) are the protocol of ``ShardModel`` on top of
the same launches, so the engines, ``prefill`` and ``generate`` drive either model class.

Precision: the residual stream, norms, routing, attention weights, decays, step sizes and recurrent
states are float32; matrix operands and the cache have the model's element type - bf16 as served, or
float32 throughout (``dtype=torch.float32``).

Launches of a layer (rows R of the step):
  R <= 16   the projection of all the mixer's parts as one GEMV; per part: attention (with norm and
            cache append inside when every row is a single token) or the recurrence's step and gated
            norm; the output projections of all parts as one GEMV; a dense feed-forward as a gated
            pair and a down GEMV, or router GEMV, gated experts + shared expert in one launch that
            also routes, weighted down-projections in one launch.  The norms of a sublayer's output,
            its residual sum and the norm of the next input run inside the next product (up to 4 rows)
            or as a launch of their own
            Latent attention: the queries' second matrix, its products per head on both sides of the attention;
            a token's vector behind a layer: its gate and its projection
            Attention with a convolution in front, or means of blocks behind its window: the same one launch in a
            step of single tokens
  R > 16    the same with GEMMs, the experts grouped by expert, their weighted sum inside the
            norm + residual launch; portions of prompts take the tiled attention and the chunked
            recurrence, single tokens beside them the split attention and the step; rotations, convolutions and
            means of blocks are launches ahead of the attention
"""

from __future__ import annotations

import numpy as np
import torch

from . import dense_ops as D
from . import ops
from .dense_ops import pad64, padded
from .model import DecoderShard
from .paged_cache import PAGE, PagedKVCache, pages_for
from .stack_config import LatentSpec, MoeSpec, StackConfig, attention_of, pooled_shape, recurrence_of, state_shape
from .stack_layers import Layer, pad8
from .state_pool import StateShape


class _Buffers:
    """Activations of up to ``rows`` rows.  The columns between a logical size and its row stride
    are zero for good: no kernel writes them."""

    def __init__(self, model: "StackModel", rows: int, seqs: int):
        self.model, self.cap = model, rows
        H, dev, t = model.cfg.hidden_size, model.device, model.dtype
        self._z = lambda *s, dtype=t: torch.zeros(*s, dtype=dtype, device=dev)  # noqa: E731
        self._named: dict[tuple, torch.Tensor] = {}
        self.tokens = self._z(rows, dtype=torch.int32)
        # the residual stream; two buffers, since a launch that also advances it reads one and
        # writes the other (``h`` is the current one)
        self.hs = [self._z(rows, H, dtype=torch.float32) for _ in range(2 if rows <= D.POST_MAX_ROWS else 1)]
        self.cur = 0
        self.xb = self._z(rows, pad64(H))                    # its copy as matrix operand
        self.xn = self._z(rows, pad64(H))                    # rows entering the head
        self.branch = self._z(rows, H, dtype=torch.float32)  # a sublayer's output
        self.branch2 = self._z(rows, H, dtype=torch.float32) if model.two_branches else None
        self.experts: dict[tuple[int, int], D.ExpertRows] = {}
        self.values: dict[int, torch.Tensor] = {}  # of layers whose values later layers mix in
        # outputs of a single-token step (last shard)
        self.logits = self.logits16 = None
        self.next_token = self._z(seqs, dtype=torch.int32)
        self.lse = self._z(seqs, dtype=torch.float32)
        self.logprob = self._z(seqs, dtype=torch.float32)
        self.argmax_ws = ops.argmax_workspace(seqs, dev)

    @property
    def h(self) -> torch.Tensor:
        return self.hs[self.cur]

    def _get(self, name: str, *shape: int, dtype=None) -> torch.Tensor:
        key = (name, *shape)
        if key not in self._named:
            self._named[key] = self._z(*shape, dtype=self.model.dtype if dtype is None else dtype)
        return self._named[key]

    def f32(self, name: str, n: int) -> torch.Tensor:
        return self._get(name, self.cap, n, dtype=torch.float32)

    def cols(self, name: str, n: int) -> torch.Tensor:
        return self._get(name, self.cap, n)

    def mixed(self, name: str, n: int) -> torch.Tensor:
        """Rows of n columns that enter a product."""
        return self._get(name, self.cap, pad64(n))

    def router_logits(self, n: int) -> torch.Tensor:
        return self._get("router", self.cap, n, dtype=torch.float32)

    def idx(self, top: int) -> torch.Tensor:
        return self._get("idx", self.cap, top, dtype=torch.int32)

    def wt(self, top: int) -> torch.Tensor:
        return self._get("wt", self.cap, top, dtype=torch.float32)

    def act(self, top: int, ff: int) -> torch.Tensor:
        return self._get(f"act{ff}", self.cap, top, pad64(ff))

    def shared_act(self, ff: int) -> torch.Tensor:
        return self._get(f"shared{ff}", self.cap, pad64(ff))

    def expert_out(self, top: int) -> torch.Tensor:
        return self._get("expert_out", self.cap, top, self.model.cfg.hidden_size)

    def shared_out(self) -> torch.Tensor:
        return self._get("shared_out", self.cap, self.model.cfg.hidden_size)


class _LatentRows:
    """A step's rows as latent attention takes them: portions over expanded keys (``pages`` to gather, ``blocks`` of
    tokens), the other rows one by one (``rows``)."""

    def __init__(self, pages, n_pages: int, blocks, n_blocks: int, rows, n_rows: int):
        self.lists, self.n_blocks, self.rows, self.n_rows = (blocks, n_blocks, pages, n_pages), n_blocks, rows, n_rows


class _Batch:
    """What the mixers need to know about the rows of a step, on the device."""

    def __init__(self, rows: int, slot, pos, keys: int, single=None, n_single: int | None = None, blocks=None,
                 want=None, n_want: int | None = None, chunks=None, n_chunks: int = 0, seqs=None, n_seqs: int = 0,
                 alone=None, n_alone: int = 0, latent: _LatentRows | None = None, means=None):
        self.rows, self.slot, self.pos, self.keys = rows, slot, pos, keys
        self.single, self.n_single = single, rows if n_single is None else n_single  # rows alone (None: all)
        self.blocks = blocks or {}                                                   # tokens -> (list, count)
        self.want, self.n_want = want, rows if n_want is None else n_want            # rows with logits
        # recurrences: portions of several tokens, cut into chunks; rows that are a portion by themselves
        self.chunks, self.n_chunks, self.seqs, self.n_seqs = chunks, n_chunks, seqs, n_seqs
        self.alone, self.n_alone, self.latent = alone, n_alone, latent
        self.means = means or {}  # positions of a block -> (list, count) of the blocks that the step completes

    @property
    def decode(self) -> bool:
        """Every row is a single token of a sequence of its own."""
        return self.n_single == self.rows and not self.blocks and self.single is None


class StackModel(DecoderShard):
    def __init__(self, cfg: StackConfig, weights: dict[str, torch.Tensor], start_layer: int = 0,
                 end_layer: int | None = None, device="cuda:0", dtype=torch.bfloat16):
        if dtype not in (torch.bfloat16, torch.float32):
            raise ValueError(f"element type {dtype} not supported (bfloat16, float32)")
        self.cfg, self.dtype, self.device = cfg, dtype, torch.device(device)
        self.start_layer = start_layer
        self.end_layer = cfg.num_hidden_layers if end_layer is None else end_layer
        if not (0 <= self.start_layer < self.end_layer <= cfg.num_hidden_layers):
            raise ValueError(f"bad layer range [{start_layer},{end_layer}) of {cfg.num_hidden_layers}")
        H, side = cfg.hidden_size, None
        if cfg.side_dim is not None:
            if not self.is_first:
                raise ValueError(f"{cfg.architecture}: every layer reads the tokens, a shard must start at layer 0")
            t = weights["side.embed"]
            if tuple(t.shape) != (cfg.vocab_size, cfg.num_hidden_layers * cfg.side_dim):
                raise ValueError(f"side.embed: shape {tuple(t.shape)}, config says {cfg.vocab_size} x {cfg.num_hidden_layers} parts of "
                                 f"{cfg.side_dim}")
            side = (cfg.side_dim, t.to(self.device, dtype).contiguous())
        self.layers = [Layer(cfg.layers[i], weights, i, H, cfg.norm, dtype, self.device, side)
                       for i in range(self.start_layer, self.end_layer)]
        self.mixed_from = {m.v_mix_from for m in (attention_of(L.spec.mixer) for L in self.layers) if m is not None and m.v_mix}
        latents = [L.spec.mixer for L in self.layers if isinstance(L.spec.mixer, LatentSpec)]
        self.has_latent, self.expands = bool(latents), all(map(D.latent_expands, latents))
        self.two_branches = any(len(L.parts) > 1 for L in self.layers)
        # layer -> index of the pool's layer that holds its keys and values, its recurrent state
        self.kv_index: dict[int, int] = {}
        self.kv_shapes: list[tuple[int, int, int]] = []
        self.kv_blocks: list[int | None] = []
        self.state_index: dict[int, int] = {}
        self.state_shapes: list[StateShape] = []
        self.recurs = any(recurrence_of(L.spec.mixer) is not None for L in self.layers)
        for L in self.layers:
            s = state_shape(L.spec.mixer)
            if s is not None:
                self.state_index[L.index] = len(self.state_shapes)
                self.state_shapes.append(s)
            m, shape = attention_of(L.spec.mixer), pooled_shape(L.spec.mixer)
            if shape is not None:
                self.kv_index[L.index] = len(self.kv_shapes)
                self.kv_shapes.append(shape)
                self.kv_blocks.append(None if m is None else m.pool)
            if m is None:
                continue
            if m.v_mix and m.v_mix_from < self.start_layer:
                raise ValueError(f"layer {L.index} mixes in the values of layer {m.v_mix_from}, which is outside the shard "
                                 f"[{self.start_layer},{self.end_layer})")
            if m.kv_from is None:
                continue
            if m.kv_from not in self.kv_index:
                raise ValueError(f"layer {L.index} uses the keys of layer {m.kv_from}, which is outside the shard "
                                 f"[{self.start_layer},{self.end_layer})")
            else:
                self.kv_index[L.index] = self.kv_index[m.kv_from]
        self.embed = self.norm = self.head = None
        if self.is_first:
            self.embed = padded(weights["embed"].to(self.device), dtype, self.device)
        if self.is_last:
            self.norm = ((cfg.norm.offset + weights["final.norm"].to(self.device).float()) * cfg.logit_scale).contiguous()
            tied = self.embed if cfg.tied else None
            self.head = tied if tied is not None else padded(weights["embed" if cfg.tied else "head"].to(self.device), dtype, self.device)
        self._bufs: dict[tuple, _Buffers] = {}
        self._graphs: dict[tuple, tuple] = {}
        self._bound: tuple | None = None  # (cache, per layer and part the argument blocks)
        self._row_ids: dict[tuple[int, int], torch.Tensor] = {}
        self.layer_hook = None  # called with (layer index, residual rows) after every layer (eager steps)

    # ------------------------------------------------------------------ engine protocol
    mixed_steps = True  # portions of prompts and decoded tokens share a step

    def weight_bytes(self) -> int:
        ts = [t for L in self.layers for t in L.tensors()] + ([self.head] if self.is_last else [])
        return sum(t.numel() * t.element_size() for t in ts)

    def make_cache(self, batch: int = 1, max_seq: int = 4096, pool_tokens: int | None = None) -> PagedKVCache:
        return PagedKVCache(self.kv_shapes, batch, max_seq, self.device, self.dtype, pool_tokens, self.state_shapes,
                            self.kv_blocks)

    def _buffers(self, B: int, T: int) -> _Buffers:
        """Activations of B x T rows: single-token steps (T = 1) have a set per batch size - a
        captured step points at it -, everything else shares one that grows in powers of two."""
        if T == 1:
            key, rows = (B, 1), B
        else:
            key, rows = ("rows",), B * T
        bf = self._bufs.get(key)
        if bf is None or bf.cap < rows:
            cap = rows if T == 1 else max(64, 1 << (rows - 1).bit_length())
            self._bufs[key] = bf = None  # (drop the old set before the larger one is allocated)
            self._bufs[key] = bf = _Buffers(self, cap, B)
        return bf

    @staticmethod
    def _keys_hint(cache: PagedKVCache, rsl: slice) -> int:
        """Upper bound (a power of two) of the keys the longest row holds after the step: launches
        are laid out for it, and a captured step stays valid below it."""
        return max(256, 1 << max(cache.offsets[rsl]).bit_length())

    def _sampling_logits(self, logits: torch.Tensor, bf: _Buffers) -> torch.Tensor:
        if logits.dtype == torch.bfloat16:
            return logits
        if bf.logits16 is None:
            bf.logits16 = torch.empty_like(logits, dtype=torch.bfloat16)
        bf.logits16.copy_(logits)
        return bf.logits16

    def _mixers(self, cache: PagedKVCache) -> list[list]:
        """Per layer, the bound operator of each part of its mixer."""
        if self._bound is None or self._bound[0] is not cache:
            self._bound = (cache, [[p.bind(cache, self.kv_index.get(L.index), self.state_index.get(L.index), self.dtype, self.cfg.eps)
                                    for p in L.parts] for L in self.layers])
        return self._bound[1]

    # ------------------------------------------------------------------ the launches
    def _settle(self, bf: _Buffers, n: int, due: D.Branches | None, pre: torch.Tensor | None) -> None:
        """residual += normed sublayer output, if one is still outstanding (``due``); bf.xb <- the
        residual, or its norm (``pre``)"""
        if due is not None:
            D.post_norm_add(due, self.cfg.eps, bf.h, bf.xb, n, pre)
        elif pre is not None:
            D.norm_rows(bf.h, pre, self.cfg.eps, bf.xb, n)

    def _product(self, bf: _Buffers, n: int, due: D.Branches | None, pre, w, out, bias=None, tail=None, up=None, spec=None,
                 keep_operand: bool = False, after: D.After | None = None) -> None:
        """out <- operand @ w^T (or the gated pair), after the outstanding norms and sum;
        ``keep_operand``: bf.xb is read by later launches too"""
        if due is not None and len(bf.hs) > 1 and D.post_linear_fits(n, w, bf.xb, self.cfg.hidden_size, pre is not None):
            x = bf.h
            bf.cur ^= 1
            D.post_linear(x, due, self.cfg.eps, bf.h, bf.xb if keep_operand else None, w, out, n, bias, tail, pre, up, spec, after)
            return
        self._settle(bf, n, due, pre)
        if up is not None:
            D.glu(bf.xb, w, up, out, n, spec)
        else:
            D.linear(bf.xb, w, out, n, bias=bias, tail=tail, after=after)

    def _mixer(self, L: Layer, bound: list, bf: _Buffers, b: _Batch, due: D.Branches | None) -> D.Branches:
        """The mixer of the residual; returns its output on the way into the residual"""
        n, eps = b.rows, self.cfg.eps
        p, mixed = L.parts[0], L.index in self.mixed_from
        y2 = bf.f32("proj_tail", pad8(L.n_tail)) if L.n_tail else None
        if L.n_main:  # (a layer whose values others mix in keeps its columns to itself)
            y = bf.cols("proj_kept" if mixed else "proj", pad8(L.n_main))
            self._product(bf, n, due, L.pre1, L.proj, y, bias=L.proj_b, tail=(y2, L.n_tail) if L.n_tail else None)
        else:
            y = None
            self._product(bf, n, due, L.pre1, L.proj, y2, bias=L.proj_b)
        if mixed:
            bf.values[L.index] = y[:, p.col + p.v_col :]
        outs = [p.run(op, bf, b, y, y2, eps) for p, op in zip(L.parts, bound)]
        if len(L.parts) == 1:
            D.linear(outs[0], p.o, bf.branch, n, bias=p.o_b)
            return D.Branches(bf.branch, L.norm1, self.cfg.norm.mult, norm=self.cfg.norm)
        D.linear_pair(outs[0], p.o, bf.branch, outs[1], L.parts[1].o, bf.branch2, n)
        return D.Branches(bf.branch, L.norm1, self.cfg.norm.mult, bf.branch2, L.gain_a, L.gain_b)

    def _dense(self, L: Layer, bf: _Buffers, n: int, due: D.Branches) -> D.Branches:
        f = L.spec.mlp
        act = bf.mixed("ff", f.ff)
        if L.ff.gate is None:
            self._product(bf, n, due, L.pre2, L.ff.up, act, after=L.ff.after)
        else:
            self._product(bf, n, due, L.pre2, L.ff.gate, act, up=L.ff.up, spec=f)
        D.linear(act, L.ff.down, bf.branch, n)
        return D.Branches(bf.branch, L.norm2, self.cfg.norm.mult, norm=self.cfg.norm)

    def _side(self, L: Layer, bf: _Buffers, n: int, due: D.Branches | None) -> D.Branches:
        """The tokens' vectors, gated by the residual: gelu(gate x) * vector, projected; then normed and added"""
        s = L.side
        act = bf.mixed("side", self.cfg.side_dim)
        self._product(bf, n, due, None, s.gate, act, after=D.After("gelu_tanh", s.table, bf.tokens))
        D.linear(act, s.proj, bf.branch, n)
        return D.Branches(bf.branch, s.gain)

    def _moe(self, L: Layer, bf: _Buffers, n: int, due: D.Branches) -> D.Branches | None:
        """The experts of the residual: bf.branch, or already normed and added (returns None)"""
        f, H, w = L.spec.mlp, self.cfg.hidden_size, L.ff
        r, mult = f.router, self.cfg.norm.mult
        logits, idx, wt = bf.router_logits(w.router.shape[0]), bf.idx(r.top), bf.wt(r.top)
        self._product(bf, n, due, L.pre2, w.router, logits, bias=w.router_b, keep_operand=True)
        if n <= D.GEMV_MAX_ROWS:
            key = (L.index, bf.cur)
            if key not in bf.experts:
                bf.experts[key] = D.ExpertRows(f, w, bf, H, bf.h)
            bf.experts[key].glu(n)
            bf.experts[key].down(n)
            return D.Branches(bf.branch, L.norm2, mult, norm=self.cfg.norm)
        D.moe_route(logits, w.correction, r.scale, idx, wt, n, r.renorm)
        act, out = bf.act(r.top, f.expert.ff), bf.expert_out(r.top)
        ws = ops.moe_group(idx[:n], r.experts, check_indices=False)  # identity ids are past the end: left out
        D.grouped_gemm(bf.xb, w.gate, ws, act, n, r.top, up=w.up, spec=f.expert)
        D.grouped_gemm(act, w.down, ws, out, n, r.top, x_per_pair=True)
        shared = None
        if f.shared is not None:
            sact, shared = bf.shared_act(f.shared.ff), bf.shared_out()
            D.glu_gemm(bf.xb, w.s_gate, w.s_up, sact, n, f.shared)
            D.linear(sact, w.s_down, shared, n)
        D.moe_sum_post_norm(out, idx, wt, shared, logits, r.experts, w.gate_col, L.norm2, self.cfg.eps, bf.h, bf.xb, n, mult,
                            self.cfg.norm)
        return None

    def _forward(self, cache: PagedKVCache, bf: _Buffers, b: _Batch, logits: bool) -> torch.Tensor:
        """Launch the shard over the rows of ``b``: input bf.tokens (first shard) or bf.hs[0]; returns
        the logits [n_want, V] of the wanted rows, or the residual."""
        n, H, eps = b.rows, self.cfg.hidden_size, self.cfg.eps
        bf.cur = 0
        if self.is_first:
            D.embed_rows(bf.tokens[:n], self.embed, bf.h, bf.xb, H, self.cfg.embed_scale)
        else:
            bf.xb[:n, :H].copy_(bf.h[:n])
        due = None  # the latest sublayer's output, which still has to pass its norm
        for L, bound in zip(self.layers, self._mixers(cache)):
            due = self._mixer(L, bound, bf, b, due)
            if L.ff is not None:
                due = (self._moe if isinstance(L.spec.mlp, MoeSpec) else self._dense)(L, bf, n, due)
            if L.side is not None:
                due = self._side(L, bf, n, due)
            if self.layer_hook is not None:
                self._settle(bf, n, due, None)
                due = None
                self.layer_hook(L.index, bf.h[:n])
        self._settle(bf, n, due, None)
        if not self.is_last or not logits:
            if bf.cur:  # callers find the residual where they put it
                bf.hs[0][:n].copy_(bf.h[:n])
                bf.cur = 0
            return bf.h[:n]
        D.norm_rows(bf.h, self.norm, eps, bf.xn, b.n_want, rows=b.want, center=self.cfg.norm.center)
        if bf.logits is None or bf.logits.shape[0] != b.n_want:
            bf.logits = torch.empty(b.n_want, self.cfg.vocab_size, dtype=self.dtype, device=self.device)
            bf.logits16 = None
        cap = self.cfg.logit_cap
        D.linear(bf.xn, self.head, bf.logits, b.n_want, after=None if cap is None else D.After("cap", cap=cap))
        bf.cur = 0
        return bf.logits

    def _run(self, B: int, T: int, cache: PagedKVCache, bf: _Buffers, logits_mode: str, rows: slice | None = None):
        """The single-token step of cache rows ``rows`` (default the first B): positions are read on
        the device, so a captured launch sequence can be replayed."""
        assert T == 1
        rsl = rows if rows is not None else slice(0, B)
        key = (rsl.start, B)
        if key not in self._row_ids:
            self._row_ids[key] = torch.arange(rsl.start, rsl.start + B, dtype=torch.int32, device=self.device)
        b = _Batch(B, self._row_ids[key], cache.pos[rsl], self._keys_hint(cache, rsl))
        return self._forward(cache, bf, b, logits_mode != "none")

    # ------------------------------------------------------------------ steps
    def _batch(self, cache: PagedKVCache, counts: list[tuple[int, int]], want: list[int]) -> _Batch:
        """``counts``: (cache row, tokens) per entry, in batch order; ``want``: batch rows with logits."""
        n = sum(c for _, c in counts)
        slot, pos, single = np.empty(n, np.int32), np.empty(n, np.int32), []
        sizes = {D.PagedAttention.prompt_block(m) for m in (attention_of(L.spec.mixer) for L in self.layers) if m is not None}
        blocks: dict[int, list] = {s: [] for s in sizes}
        chunks, seqs, alone = [], [], []
        pages, lat_blocks, lat_rows = [], [], []  # latent attention
        means: dict[int, list] = {p: [] for p in self.kv_blocks if p}
        C = D.recur_chunk() if self.recurs else 0
        at, keys = 0, 1
        tiled = self.dtype == torch.bfloat16  # the 32-bit mode runs every position by itself
        for row, c in counts:
            p0 = cache.offsets[row]
            slot[at : at + c] = row
            pos[at : at + c] = np.arange(p0, p0 + c)
            keys = max(keys, p0 + c)
            if c == 1 or not tiled:
                single.extend(range(at, at + c))
            else:
                for s in sizes:
                    blocks[s] += [(at + o, row, p0 + o, min(s, c - o)) for o in range(0, c, s)]
            if self.has_latent and self.expands and tiled and c >= D.LATENT_SHORT:
                lat_blocks += [(at + o, len(pages) * PAGE, p0 + o, min(D.LATENT_BLOCK, c - o)) for o in range(0, c, D.LATENT_BLOCK)]
                pages += [(row, i) for i in range(pages_for(p0 + c))]
            elif self.has_latent:
                lat_rows.extend(range(at, at + c))
            for p, blks in means.items():
                blks += [(row, i) for i in range(p0 // p, (p0 + c) // p)]
            if C and c == 1:
                alone.append(at)
            elif C:
                seqs.append((len(chunks), -(-c // C), 0, 0))
                chunks += [(at + o, row, p0 + o, min(C, c - o), p0, 0, 0, 0) for o in range(0, c, C)]
            at += c
        parts = [slot, pos] + [np.asarray(x, np.int32).reshape(-1) for x in (single, want, chunks, seqs, alone, pages, lat_blocks, lat_rows)]
        have = [s for s in sizes if blocks[s]]
        parts += [np.asarray(blocks[s], np.int32).reshape(-1) for s in have]
        parts += [np.asarray(x, np.int32).reshape(-1) for x in means.values()]
        starts, total = [], 0
        for p in parts:  # 16-byte aligned pieces of one upload
            starts.append(total)
            total += -(-p.size // 4) * 4
        flat = np.zeros(total, np.int32)
        for s0, p in zip(starts, parts):
            flat[s0 : s0 + p.size] = p
        dev = torch.empty(total, dtype=torch.int32, device=self.device)
        ops.put_ints(dev, flat)
        t = [dev[s0 : s0 + p.size] for s0, p in zip(starts, parts)]
        latent = _LatentRows(t[7], len(pages), t[8], len(lat_blocks), t[9], len(lat_rows)) if self.has_latent else None
        one_each = all(c == 1 for _, c in counts)
        return _Batch(n, t[0], t[1], keys, single=None if one_each else t[2], n_single=len(single),
                      blocks={s: (t[10 + i], len(blocks[s])) for i, s in enumerate(have)},
                      want=t[3], n_want=len(want), chunks=t[4], n_chunks=len(chunks), seqs=t[5], n_seqs=len(seqs),
                      alone=t[6], n_alone=len(alone), latent=latent,
                      means={p: (t[10 + len(have) + i], len(x)) for i, (p, x) in enumerate(means.items())})

    def step(self, cache: PagedKVCache, entries: list[tuple[int, list[int], list[int]]]) -> torch.Tensor | None:
        """One batch: ``entries`` are (cache row, its next tokens, places among them whose logits are
        asked for), each row at most once.  Appends the tokens to the rows' sequences and returns
        the logits [wanted, V] in entry order (None if nothing is wanted).  The result is valid until
        the next step, and on the current stream, as any tensor's contents: the call returns before the launches have run."""
        if not (self.is_first and self.is_last):
            raise ValueError("step() needs a shard that holds the whole model")
        if len({e[0] for e in entries}) != len(entries) or any(not e[1] for e in entries):
            raise ValueError("a step takes each row once, with at least one token")
        V = self.cfg.vocab_size
        tokens = [int(t) for _, toks, _ in entries for t in toks]
        if tokens and not 0 <= min(tokens) <= max(tokens) < V:
            raise ValueError(f"token ids outside [0, {V})")
        want, at = [], 0
        for _, toks, places in entries:
            if any(not 0 <= w < len(toks) for w in places):
                raise ValueError(f"places {places} outside a portion of {len(toks)} tokens")
            want += [at + w for w in places]
            at += len(toks)
        return self._step(cache, [(r, len(t)) for r, t, _ in entries], want, tokens=tokens)

    def _step(self, cache, counts, want, tokens=None, hidden=None) -> torch.Tensor | None:
        n = sum(c for _, c in counts)
        if n == 0:
            return None
        cache.order()
        cache.reserve_each(counts)
        bf = self._buffers(1, max(n, 2))
        if tokens is not None:
            ops.put_ints(bf.tokens[:n], tokens)
        else:
            bf.h[:n].copy_(hidden)
        b = self._batch(cache, counts, want)
        out = self._forward(cache, bf, b, bool(want))
        for row, c in counts:
            cache.advance_host(c, [row])
        cache.sync_pos()
        return out if want or not self.is_last else None

    def __call__(self, tokens: torch.Tensor | None, cache: PagedKVCache,
                 input_embeddings: torch.Tensor | None = None, logits: str = "all",
                 rows: slice | None = None) -> torch.Tensor:
        """``ShardModel.__call__``: tokens int [B,T] (first shard) or input_embeddings float32 [B,T,H];
        appends T entries to the cache rows; logits [B,T,V] ("all"), [B,1,V] ("last") on the last
        shard, else the residual [B,T,H] (float32)."""
        src = tokens if self.is_first else input_embeddings
        assert src is not None
        B, T = src.shape[:2]
        r0 = rows.start if rows is not None else 0
        if (rows is not None and rows.stop - rows.start != B) or r0 + B > cache.batch:
            raise ValueError(f"batch {B} does not match cache rows {rows} (cache batch {cache.batch})")
        want: list[int] = []
        if self.is_last and logits != "none":
            want = list(range(B * T)) if logits == "all" else [b * T + T - 1 for b in range(B)]
        counts = [(r0 + b, T) for b in range(B)]
        if self.is_first:
            out = self._step(cache, counts, want, tokens=tokens.reshape(-1).tolist())
        else:
            out = self._step(cache, counts, want, hidden=input_embeddings.reshape(B * T, -1))
        if want:
            return out.view(B, -1, self.cfg.vocab_size).clone()
        return self._bufs[("rows",)].h[: B * T].view(B, T, -1).clone()
