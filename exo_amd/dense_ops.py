"""Operators of the layer-list decoders on torch device tensors (C ABI of include/exo_mi355x.h):
products with unquantised matrices, residual norms, routing, experts, attention over a paged pool
and recurrences over a state pool.  Element type bf16 or float32 throughout (the tensors' dtype decides); like ``ops``, every
function launches on torch's current stream and never synchronises.

Matrix operands have row strides of multiples of 64 elements with zeros past the logical size
(``padded``): no kernel has a tail in K.
"""

from __future__ import annotations

import ctypes as C

import torch

from . import native
from .native import check
from .ops import _ptr, _stream

GEMV_MAX_ROWS = 16


def pad64(n: int) -> int:
    return -(-n // 64) * 64


def padded(w: torch.Tensor, dtype, device) -> torch.Tensor:
    """[..., N, K] -> contiguous [..., N, pad64(K)] of ``dtype`` with zeros behind K."""
    out = torch.zeros(*w.shape[:-1], pad64(w.shape[-1]), dtype=dtype, device=device)
    out[..., : w.shape[-1]].copy_(w)
    return out


def _code(t: torch.Tensor) -> int:
    if t.dtype == torch.bfloat16:
        return 0
    if t.dtype == torch.float32:
        return 1
    raise ValueError(f"element type {t.dtype} not supported (bfloat16, float32)")


def embed_rows(ids, table, x, xb, H: int, scale: float = 1.0) -> None:
    n = ids.numel()
    check(native.load().exo_embed_rows(_ptr(ids), _ptr(table), _ptr(x), _ptr(xb), n, table.shape[0], H,
                                       table.shape[1], xb.shape[1], scale, _code(xb), _stream()), "embed_rows")


def norm_rows(x, gain, eps: float, out, n: int, rows=None, center: bool = False) -> None:
    """out[i] = x[i] (rows: x[rows[i]]) / rms * gain; ``center``: its mean is taken off first."""
    check(native.load().exo_norm_rows(x.data_ptr(), _ptr(rows), _ptr(gain), _ptr(out), n, gain.numel(), x.stride(0),
                                      out.shape[1], eps, int(center), _code(out), _stream()), "norm_rows")


def _p(t):
    return None if t is None else t.data_ptr()


class Branches:
    """A sublayer's output on its way into the residual: ``branch``, or half the sum of two branches that
    are normed each with a gain of its own first (``branch2``, ``gain_a``, ``gain_b``); then the norm with
    ``gain`` (None: no norm), times ``mult``.  ``norm``: a NormSpec that asks for the norm of the sum instead (the residual times
    ``norm.keep``).  All float32."""

    def __init__(self, branch, gain, mult: float = 1.0, branch2=None, gain_a=None, gain_b=None, norm=None):
        self.branch, self.gain, self.mult = branch, gain, mult
        self.branch2, self.gain_a, self.gain_b = branch2, gain_a, gain_b
        self.of_sum = norm is not None and norm.of_sum
        self.center, self.keep = self.of_sum and norm.center, norm.keep if self.of_sum else 1.0

    def args(self, x, x_out, operand, eps: float, pre) -> native.PostNorm:
        return native.PostNorm(x=_p(x), branch=_p(self.branch), branch2=_p(self.branch2), gain_a=_p(self.gain_a),
                               gain_b=_p(self.gain_b), gain=_p(self.gain), pre=_p(pre), x_out=_p(x_out),
                               operand=_p(operand), H=(x if self.gain is None else self.gain).shape[-1], ldb=0 if self.branch is None else self.branch.stride(0),
                               sum=int(self.of_sum), center=int(self.center), eps=eps, mult=self.mult, keep=self.keep)


def post_norm_add(br: Branches, eps: float, x, xb, n: int, pre=None) -> None:
    """x += the normed branches; xb = x (or its norm with gain ``pre``) in the element type."""
    check(native.load().exo_post_norm_add(C.byref(br.args(x, x, xb, eps, pre)), n, xb.shape[1],
                                          _code(xb), _stream()), "post_norm_add")


def moe_sum_post_norm(y, idx, wt, shared, logits, experts: int, gate_col: int, gain, eps: float, x, xb, n: int,
                      mult: float = 1.0, norm=None) -> None:
    """x += norm(weighted sum of the chosen experts' outputs y [n, top, ld] + shared, gated by the logits'
    ``gate_col`` unless that is negative); ``norm`` as for ``Branches``."""
    q = Branches(None, gain, mult, norm=norm).args(x, x, xb, eps, None)
    check(native.load().exo_moe_sum_post_norm(
        _ptr(y), _ptr(idx), _ptr(wt), _ptr(shared), _ptr(logits), idx.shape[1], experts, y.shape[-1],
        0 if shared is None else shared.shape[1], logits.shape[1], gate_col, C.byref(q), n, xb.shape[1], _code(xb),
        _stream()), "moe_sum_post_norm")


def moe_route(logits, correction, scale: float, idx, wt, n: int, renorm: bool = False) -> None:
    check(native.load().exo_moe_route(_ptr(logits), _ptr(correction), _ptr(idx), _ptr(wt), n, correction.numel(),
                                      logits.shape[1], idx.shape[1], scale, int(renorm), _stream()), "moe_route")


_GEMM_WS: dict[int, torch.Tensor] = {}
GEMM_WS_FLOATS = 1 << 24


def gemm_workspace(device) -> torch.Tensor:
    """Float32 partial tiles of single products that split K; one per device (work is in stream order)."""
    key = torch.device(device).index or 0
    if key not in _GEMM_WS:
        _GEMM_WS[key] = torch.empty(GEMM_WS_FLOATS, dtype=torch.float32, device=device)
    return _GEMM_WS[key]


def pair_workspace(a, device):
    """... of a gated pair, for this launch alone: pairs on two streams may run side by side."""
    need = native.load().exo_linear_pair_workspace(C.byref(a))
    return torch.empty(need, dtype=torch.float32, device=device) if need else None


ACTS = {None: 0, "relu2": 1, "gelu_tanh": 2, "cap": 3}


class After:
    """What happens to a product's result ahead of its store: ``act`` (cap: bent at +-``cap``), then times row
    ``rows[m]`` (or m) of ``mul`` (element type)."""

    def __init__(self, act: str | None = None, mul=None, rows=None, cap: float = 0.0):
        self.act, self.mul, self.rows, self.cap = act, mul, rows, cap


def _linear(x, w, out, n: int, bias=None, tail=None, up=None, spec=None, after: After | None = None) -> native.Linear:
    """``tail``: float32 output of the columns past ``out``'s share (w's rows beyond N - tail's logical
    columns; given as (tensor, columns)).  ``up``, ``spec``: the gated pair."""
    N = w.shape[0]
    t, nt = (None, 0) if tail is None else tail
    f = after or After()
    return native.Linear(
        x=_p(x), w=w.data_ptr(), w_up=_p(up), bias=_p(bias), y=out.data_ptr(), y2=_p(t), M=n, N=N, n1=N - nt,
        ldx=w.shape[1] if x is None else x.stride(0), ldw=w.shape[1], ldy=out.stride(0), ldy2=0 if t is None else t.stride(0),
        y_f32=int(out.dtype == torch.float32), dtype=_code(w), limit=spec.limit if spec else 0.0,
        alpha=spec.alpha if spec else 0.0, shift=spec.shift if spec else 0.0, cubic=spec.cubic if spec else 0.0, cap=f.cap,
        act=ACTS[f.act], mul=_p(f.mul),
        mul_rows=_p(f.rows), ldmul=0 if f.mul is None else f.mul.stride(0))


def linear(x, w, out, n: int, bias=None, force_gemm: bool = False, tail=None, after: After | None = None) -> None:
    """out[:n] = x[:n] @ w^T (+ bias float32); out in x's element type or float32.  ``tail`` (tensor, columns):
    the last columns go to that float32 tensor instead."""
    _launch_linear(_linear(x, w, out, n, bias, tail, after=after), n, x.device, force_gemm)


def _launch_linear(a, n: int, device, force_gemm: bool = False) -> None:
    if n <= GEMV_MAX_ROWS and not force_gemm:
        check(native.load().exo_linear_rows(C.byref(a), None, _stream()), "linear")
    else:
        ws = pair_workspace(a, device) if a.w_up else gemm_workspace(device)
        check(native.load().exo_linear_gemm(C.byref(a), _ptr(ws), 0 if ws is None else ws.numel(), _stream()), "linear(gemm)")


def linear_pair(x0, w0, out0, x1, w1, out1, n: int) -> None:
    """Two products over the same number of rows: one launch for few rows."""
    a, b = _linear(x0, w0, out0, n), _linear(x1, w1, out1, n)
    if n <= GEMV_MAX_ROWS:
        check(native.load().exo_linear_rows(C.byref(a), C.byref(b), _stream()), "linear_pair")
    else:
        _launch_linear(a, n, x0.device)
        _launch_linear(b, n, x1.device)


POST_MAX_ROWS = 4  # (rows of a buffer set that keeps two residuals)


def post_linear_fits(n: int, w, xb, H: int, pre: bool = False) -> bool:
    """Whether (and by measurement) the norms belong inside the product: every workgroup repeats them."""
    if n * H > 4096 or (pre and H > 2048):
        return False
    return n <= POST_MAX_ROWS and bool(native.load().exo_post_linear_fits(n, w.shape[0], H, xb.shape[1], _code(xb)))


def post_linear(x, br: Branches, eps: float, x_out, xb, w, out, n: int, bias=None, tail=None, pre=None, up=None,
                spec=None, after: After | None = None) -> None:
    """``post_norm_add`` and ``linear`` (or the gated pair) in one launch: x_out = x + the normed branches
    (another buffer than x), xb (may be None) the product's operand.  x and x_out None: the normed branch
    alone is the operand."""
    q, a = br.args(x, x_out, xb, eps, pre), _linear(None, w, out, n, bias, tail, up, spec, after)
    check(native.load().exo_post_linear(C.byref(q), C.byref(a), _stream()), "post_linear")


def norm_linear(x, gain, eps: float, operand, w, out, n: int) -> None:
    """out[:n] = (x / rms * gain) @ w^T, x float32 rows; ``operand``: scratch for the normed rows."""
    br = Branches(x, gain)
    fits = n <= GEMV_MAX_ROWS and n * gain.numel() <= 4096 and native.load().exo_post_linear_fits(
        n, w.shape[0], gain.numel(), operand.shape[1], _code(operand))  # (no residual: any rows of a GEMV)
    if fits:
        post_linear(None, br, eps, None, None, w, out, n)
    else:
        norm_rows(x, gain, eps, operand, n)
        linear(operand, w, out, n)


def glu(x, gate, up, out, n: int, spec, force_gemm: bool = False) -> None:
    """out[:n] = clamped gated unit of x[:n].  (Pairs of few tiles take a buffer of partial sums from torch's allocator, on its
    current stream.)"""
    _launch_linear(_linear(x, gate, out, n, up=up, spec=spec), n, x.device, force_gemm)


def glu_gemm(x, gate, up, out, n: int, spec) -> None:
    glu(x, gate, up, out, n, spec, force_gemm=True)


def grouped_gemm(x, w, group_ws, out, T: int, topk: int, up=None, spec=None, x_per_pair: bool = False) -> None:
    """Experts w [E, N, K] over (token, slot) pairs sorted by ``ops.moe_group``: out row = pair.
    ``up`` and ``spec``: the gated pair."""
    lim, al, sh = (spec.limit, spec.alpha, spec.shift) if up is not None else (0.0, 0.0, 0.0)
    check(native.load().exo_dense_grouped_gemm(
        _ptr(x), _ptr(w), _ptr(up), _ptr(group_ws), _ptr(out), lim, al, sh, T, topk, int(x_per_pair), w.shape[0],
        w.shape[1], x.shape[-1], w.shape[2], out.shape[-1], _code(x), _stream()), "grouped_gemm")


class ExpertRows:
    """The experts of a decode step (up to 16 rows): argument block built once per layer and
    residual buffer, launched as gated products (which also route) and as weighted down-projections."""

    def __init__(self, moe, w, bf, H: int, h):
        """``moe``: MoeSpec; ``w``: the layer's tensors; ``bf``: the activation buffers; ``h``: the
        residual that enters the feed-forward."""
        r, e, s = moe.router, moe.expert, moe.shared
        p = lambda t: None if t is None else t.data_ptr()  # noqa: E731
        self.args = native.MoeRows(
            x=p(bf.xb), gate=p(w.gate), up=p(w.up), down=p(w.down),
            shared_gate=p(w.s_gate), shared_up=p(w.s_up), shared_down=p(w.s_down),
            act=p(bf.act(r.top, e.ff)), shared_act=p(bf.shared_act(s.ff)) if s else None, out=p(bf.branch),
            x_res=p(h), idx=p(bf.idx(r.top)), wt=p(bf.wt(r.top)), logits=p(bf.router_logits(w.router.shape[0])),
            correction=p(w.correction),
            top=r.top, experts=r.experts, ff=e.ff, shared_ff=s.ff if s else 0, H=H, ldx=bf.xb.shape[1],
            lda=pad64(e.ff), ldsa=pad64(s.ff) if s else 0, ldl=w.router.shape[0], gate_col=w.gate_col, outputs=r.outputs,
            renorm=int(r.renorm), router_scale=r.scale,
            dtype=_code(bf.xb), limit=e.limit, alpha=e.alpha, shift=e.shift,
            shared_limit=s.limit if s else 0.0, shared_alpha=s.alpha if s else 0.0, shared_shift=s.shift if s else 0.0)

    def glu(self, n: int) -> None:
        self.args.rows = n
        check(native.load().exo_moe_glu_rows(C.byref(self.args), _stream()), "moe_glu_rows")

    def down(self, n: int) -> None:
        self.args.rows = n
        check(native.load().exo_moe_down_rows(C.byref(self.args), _stream()), "moe_down_rows")


_ATTN_WS: dict[int, list[torch.Tensor]] = {}


def attn_workspace(n: int, heads: int, vdim: int, nsplit: int, device) -> torch.Tensor:
    """Partials and arrival counters of split decode attention, one per device, grown on demand (a
    replaced buffer stays alive: a captured graph may point at it)."""
    need = native.load().exo_paged_attn_workspace(n, heads, vdim, nsplit)
    key = torch.device(device).index or 0
    have = _ATTN_WS.setdefault(key, [])
    if not have or have[-1].numel() < need:
        have.append(torch.zeros(need, dtype=torch.uint8, device=device))  # counters start at zero
    return have[-1]


class PagedAttention:
    """Attention of one layer over a paged pool.  ``spec``: AttentionSpec; ``li``: index of the
    pool's layer that holds its keys and values; ``freq``: float64 turns per position of each rotated pair;
    ``weight_bias``: of sigmoid weights; ``conv_w``, ``si``: the convolution's taps [taps, channels] and the index
    of the state pool's layer with its latest inputs."""

    def __init__(self, spec, slopes, li: int, cache, eps: float, q_gain=None, k_gain=None, freq=None, weight_bias=None,
                 conv_w=None, si: int | None = None):
        self.spec, self.slopes, self.cache, self.keep = spec, slopes, cache, (q_gain, k_gain, freq, weight_bias, conv_w)
        k, v = cache.k[li], cache.v[li]
        # whether queries and keys of a step need a launch of their own ahead of prompt attention
        self.prepares = bool(spec.whole_norm or spec.rot is not None or spec.v_mix or spec.conv or spec.shared_kv)
        if spec.pool and cache.blocks[li] != spec.pool:
            raise ValueError(f"the cache keeps means of blocks of {cache.blocks[li]}, attention asks for {spec.pool}")
        means = cache.means[spec.pool].table if spec.pool else None
        self.args = native.PagedAttn(
            k_pool=k.data_ptr(), v_pool=v.data_ptr(), table=cache.table.data_ptr(),
            slopes=_p(slopes), q_gain=_p(q_gain), k_gain=_p(k_gain), scale=spec.scale, eps=eps,
            heads=spec.heads, kv_heads=spec.kv_heads, dim=spec.dim, vdim=spec.vdim, ldk=k.shape[3], ldv=v.shape[2],
            max_pages=cache.table.shape[1], window=spec.window or 0, keep_first=spec.keep_first,
            unit_qk=int(spec.unit_qk), whole_norm=int(spec.whole_norm), rot=spec.rot.dims if spec.rot else 0, freq=_p(freq),
            softcap=spec.softcap or 0.0, dtype=_code(k), rot_half=int(bool(spec.rot and spec.rot.half)),
            rot_amp=spec.rot.amplitude if spec.rot else 1.0, plus_one=int(spec.plus_one), weight_bias=_p(weight_bias),
            shared_kv=int(spec.shared_kv), pool=spec.pool or 0, mean_table=_p(means),
            mean_pages=0 if means is None else means.shape[1])
        if spec.pool:
            self.args.mean_k, self.args.mean_v = cache.mean_k[li].data_ptr(), cache.mean_v[li].data_ptr()
        if spec.conv:
            self.args.conv_w, self.args.ring, self.args.taps = conv_w.data_ptr(), cache.states.ring[si].data_ptr(), spec.conv
            self.args.map = cache.states.map.data_ptr()

    def _bind(self, qkv, out, slot, pos, lst, n: int, gate=None, prepared: bool = False, out_gate=None):
        a = self.args
        a.prepared = int(prepared and self.prepares)
        assert qkv.dtype == self.cache.k[0].dtype
        a.qkv, a.ldq, a.n = qkv.data_ptr(), qkv.stride(0), n
        a.out, a.ldo = (None, 0) if out is None else (out.data_ptr(), out.stride(0))
        a.gate, a.ldg = (None, 0) if gate is None else (gate.data_ptr(), gate.stride(0))
        a.out_gate, a.ldog = (None, 0) if out_gate is None else (out_gate.data_ptr(), out_gate.stride(0))
        a.q_out, a.ldqo = None, 0
        a.slot = None if slot is None else slot.data_ptr()
        a.pos = None if pos is None else pos.data_ptr()
        a.list = None if lst is None else lst.data_ptr()
        return C.byref(a)

    def mix_values(self, v, weight: float) -> None:
        """Own values become (1 - weight) own + weight ``v`` (element type, a row per row of the step)."""
        self.args.v_mix, self.args.ldmix, self.args.mix = v.data_ptr(), v.stride(0), weight

    def append(self, qkv, slot, pos, n: int, q_out=None, blocks=None, n_blocks: int = 0):
        """Keys and values of n rows into the pool; a design that prepares also turns the queries, in place or
        (behind a convolution) into ``q_out``, and says ``prepared`` to what follows.  ``blocks``: int32
        [n_blocks, 2], the (cache row, block) whose last position is among the rows.  Returns the rows that the
        queries are now in."""
        a = self._bind(qkv, None, slot, pos, None, n)
        if self.spec.conv:
            self.args.q_out, self.args.ldqo = q_out.data_ptr(), q_out.stride(0)
            qkv = q_out
        if self.prepares:
            check(native.load().exo_paged_prepare(a, _stream()), "paged_prepare")
        else:
            check(native.load().exo_paged_append(a, _stream()), "paged_append")
        if self.spec.pool and n_blocks:
            check(native.load().exo_paged_means(self._bind(qkv, None, slot, pos, blocks, n_blocks), _stream()), "paged_means")
        return qkv

    def visible(self, keys: int) -> int:
        """Most keys one query sees when its sequence holds ``keys``."""
        s = self.spec
        return keys if s.window is None else min(keys, s.window + s.keep_first + (keys // s.pool if s.pool else 0))

    def rows(self, qkv, out, slot, pos, n: int, keys: int, append: bool, lst=None, gate=None, out_gate=None) -> None:
        """One query position per row (``lst``: which rows, else the first n).  ``keys``: most keys
        any of the sequences holds, as the host knows it (lays out the launch).  ``gate``: float32
        [rows, heads], head h's output times its sigmoid; ``out_gate``: element type, the same per output."""
        s = self.spec
        tiles = -(-self.visible(keys) // 32) + 2
        wgs = n * s.kv_heads * (-(-(s.heads // s.kv_heads) // 16))
        nsplit = max(1, min(-(-tiles // 4), 256 // wgs, 16))
        if nsplit > 8:  # (the head groups of one split then share an XCD's L2)
            nsplit = 16 if 16 * wgs <= 256 else 8
        if n * s.heads > 16384:
            nsplit = 1
        ws = attn_workspace(n, s.heads, s.vdim, nsplit, qkv.device) if nsplit > 1 else None
        check(native.load().exo_paged_attn_rows(self._bind(qkv, out, slot, pos, lst, n, gate, not append, out_gate), nsplit, int(append), _ptr(ws),
                                                0 if ws is None else ws.numel(), _stream()), "paged_attn_rows")

    @staticmethod
    def prompt_block(spec) -> int:
        return native.load().exo_paged_prompt_block(spec.heads, spec.kv_heads)

    def prompt(self, qkv, out, blocks, n: int, gate=None, out_gate=None) -> None:
        """Portions of prompts: blocks int32 [n, 4] = first row, slot, first position, tokens."""
        check(native.load().exo_paged_attn_prompt(self._bind(qkv, out, None, None, blocks, n, gate, True, out_gate), _stream()),
              "paged_attn_prompt")


_LATENT_WS: dict[tuple, list[torch.Tensor]] = {}


def latent_workspace(kind: str, n: int, dtype, device) -> torch.Tensor:
    """Partials of split rows ("parts", float32) and expanded latents, one per kind and device, grown on
    demand (replaced partials stay alive: a captured graph may point at them)."""
    key = (kind, dtype, torch.device(device).index or 0)
    have = _LATENT_WS.setdefault(key, [])
    if not have or have[-1].numel() < n:
        if kind != "parts":
            have.clear()
        have.append(torch.empty(n, dtype=dtype, device=device))
    return have[-1][:n]


LATENT_BLOCK = 128  # tokens of a block of expanded prompt attention
LATENT_SHORT = 32   # portions below this many tokens go through the absorbed rows


def latent_expands(spec) -> bool:
    """Whether a design's expanded keys and values fit the prompt kernel (else all rows are absorbed)."""
    return -(-spec.dim // 8) + -(-spec.rot_dim // 8) <= 32 and spec.vdim <= 256


class LatentAttention:
    """Latent attention of one layer over a paged pool.  ``spec``: LatentSpec; ``w``: the layer's tensors
    (``stack_layers.LatentPart``); ``li``: index of the pool's layer."""

    def __init__(self, spec, w, li: int, cache, eps: float):
        self.spec, self.w, self.cache = spec, w, cache
        pool = cache.k[li]
        self.args = native.LatentAttn(
            gain=w.kv_gain.data_ptr(), freq=_p(w.freq), pool=pool.data_ptr(), table=cache.table.data_ptr(), scale=spec.scale,
            eps=eps, heads=spec.heads, rank=spec.kv_rank, rot=spec.rot_dim, rot_col=w.rot_col, ldk=pool.shape[3],
            max_pages=cache.table.shape[1], dtype=_code(pool))

    def _bind(self, q, kv, slot, pos, n: int, lst=None, prepared: bool = False):
        a = self.args
        a.q, a.ldq, a.kv, a.ldkv, a.n = q.data_ptr(), q.stride(0), kv.data_ptr(), kv.stride(0), n
        a.slot, a.pos, a.list, a.prepared = slot.data_ptr(), pos.data_ptr(), _p(lst), int(prepared)
        return a

    def prepare(self, q, kv, slot, pos, n: int) -> None:
        """Latents and shared key parts of n rows into the pool; the queries' rotated parts in place."""
        check(native.load().exo_latent_prepare(C.byref(self._bind(q, kv, slot, pos, n)), _stream()), "latent_prepare")

    def rows(self, q, kv, ql, ol, out, slot, pos, n: int, keys: int, append: bool, lst=None) -> None:
        """One query position per row (``lst``: which rows, else the first n): ``out`` [rows, heads * vdim].
        ``ql``, ``ol``: scratch, [rows, heads * pad64(kv_rank)]; ``keys``: most keys any sequence holds."""
        s, w, lib = self.spec, self.w, native.load()
        head_linear(q, w.nope_pad, w.uk, ql, pad64(s.kv_rank), n, s.dim, lst)
        tiles, wgs = -(-keys // 64), n * (-(-s.heads // 16))
        nsplit = max(1, min(tiles, 256 // wgs, max(16, 64 // n)))  # (more partials cost the merge what they gain here)
        a = self._bind(q, kv, slot, pos, n, lst, not append)
        a.q_latent, a.ldql, a.nsplit = ql.data_ptr(), ql.stride(0), nsplit
        parts = None
        if nsplit == 1:
            a.out, a.ldo = ol.data_ptr(), ol.stride(0)
        else:
            parts = latent_workspace("parts", lib.exo_latent_parts(n, s.heads, s.kv_rank, nsplit), torch.float32, q.device)
            a.parts, a.parts_floats = parts.data_ptr(), parts.numel()
        check(lib.exo_latent_rows(C.byref(a), int(append), _stream()), "latent_rows")
        head_linear(ol, pad64(s.kv_rank), w.uv, out, s.vdim, n, s.kv_rank, lst, parts, nsplit)

    def prompt(self, q, kv, out, slot, pos, blocks, n_blocks: int, pages, n_pages: int) -> None:
        """Portions of prompts over expanded keys and values: ``pages`` int32 [n, 2] (cache row, page of its
        sequence), ``blocks`` int32 [n, 4] (first row, first gathered key row, first position, tokens)."""
        for _, launch in self.prompt_launches(q, kv, out, slot, pos, blocks, n_blocks, pages, n_pages):
            launch()

    def prompt_launches(self, q, kv, out, slot, pos, blocks, n_blocks: int, pages, n_pages: int) -> list[tuple]:
        """The launches of ``prompt``, by name."""
        s, w, lib, dev = self.spec, self.w, native.load(), q.device
        n, H, r8 = 64 * n_pages, s.heads, -(-s.rot_dim // 8) * 8
        new = lambda kind, *shape: latent_workspace(kind, shape[0] * shape[1], torch.bfloat16, dev).view(*shape)  # noqa: E731
        c, kr = new("latents", n, pad64(s.kv_rank)), new("rotated", n, r8)
        k, v = new("keys", n, H * w.d8), new("values", H * s.vdim, n)
        a = self._bind(q, kv, slot, pos, 1)
        p = native.LatentPrompt(
            q=q.data_ptr(), k=k.data_ptr(), k_rot=kr.data_ptr(), v=v.data_ptr(), list=blocks.data_ptr(), out=out.data_ptr(),
            scale=s.scale, n=n_blocks, heads=H, vdim=s.vdim, d8=w.d8, r8=r8, ldq=q.stride(0), q_head=w.nope_pad,
            rot_col=w.rot_col, ldk=k.stride(0), ldv=v.stride(0), ldo=out.stride(0))
        return [
            ("gather", lambda: check(lib.exo_latent_gather(C.byref(a), pages.data_ptr(), n_pages, c.data_ptr(), kr.data_ptr(),
                                                           _stream()), "latent_gather")),
            ("keys", lambda: linear(c, w.uk_rows, k, n, force_gemm=True)),
            ("values", lambda: linear(w.uv_rows, c, v, H * s.vdim, force_gemm=True)),
            ("attention", lambda: check(lib.exo_latent_prompt(C.byref(p), _stream()), "latent_prompt"))]


def head_linear(x, x_head: int, w, y, y_head: int, n: int, K: int, lst=None, parts=None, nsplit: int = 1) -> None:
    """y[row][h] = w[h] x[row][h] for n rows (``lst``: which): w [heads, N, pad64(K)], head h at h * x_head and
    h * y_head; ``parts``: x is merged from the partials of split latent rows."""
    a = native.HeadLinear(
        x=x.data_ptr(), w=w.data_ptr(), parts=_p(parts), parts_floats=0 if parts is None else parts.numel(), y=y.data_ptr(),
        list=_p(lst), n=n, heads=w.shape[0], N=w.shape[1], K=K, ldx=x.stride(0), x_head=x_head, ldw=w.shape[2], ldy=y.stride(0),
        y_head=y_head, nsplit=nsplit, dtype=_code(w))
    check(native.load().exo_head_linear(C.byref(a), _stream()), "head_linear")


_RECUR_WS: dict[int, torch.Tensor] = {}


def recur_workspace(nbytes: int, device) -> torch.Tensor:
    """Scores and states of recurrences over prompts, one per device, grown on demand (work is in
    stream order; single-token steps, which are captured, do not use it)."""
    key = torch.device(device).index or 0
    if key not in _RECUR_WS or _RECUR_WS[key].numel() < nbytes:
        _RECUR_WS.pop(key, None)
        _RECUR_WS[key] = torch.empty(nbytes, dtype=torch.uint8, device=device)
    return _RECUR_WS[key]


def recur_chunk() -> int:
    return native.load().exo_recur_chunk()


class Recurrence:
    """A recurrent mixer of one layer over a state pool.  ``core``: heads, key groups, key size, value size;
    ``li``: index of the pool's layer; ``consts``: members of ``native.Recurrence`` that hold for every
    launch (tensors stand for their addresses)."""

    def __init__(self, core: tuple[int, int, int, int], li: int, cache, dtype, consts: dict):
        self.heads, self.groups, self.dim, self.vdim = core
        self.cache, self.consts = cache, consts
        st, ring, peak = (x[li] for x in (cache.states.state, cache.states.ring, cache.states.peak))
        self.args = native.Recurrence(
            heads=self.heads, groups=self.groups, dim=self.dim, vdim=self.vdim, state=st.data_ptr(), lds=st.shape[3],
            map=cache.states.map.data_ptr(), ring=_p(ring), taps=0 if ring is None else ring.shape[1],
            channels=0 if ring is None else ring.shape[2], peak=_p(peak), dtype=0 if dtype == torch.bfloat16 else 1,
            **{k: v.data_ptr() if isinstance(v, torch.Tensor) else v for k, v in consts.items()})

    def bind(self, y, **inputs) -> None:
        """Where a step's inputs and outputs lie: ``y`` float32 [rows, heads * vdim]; ``inputs``: members
        by name, tensors with their row strides (``ld`` member of the same name)."""
        a = self.args
        a.y, a.ldy = y.data_ptr(), y.stride(0)
        for name, (t, ld) in inputs.items():
            setattr(a, name, t.data_ptr())
            setattr(a, ld, t.stride(0))

    def step(self, slot, pos, n: int, lst=None) -> None:
        """Single tokens: row i (``lst``: which rows, else the first n) is of cache row slot[i] at pos[i]."""
        a = self.args
        a.slot, a.pos, a.list, a.n = slot.data_ptr(), pos.data_ptr(), _p(lst), n
        check(native.load().exo_recur_step(C.byref(a), _stream()), "recur_step")

    def chunks(self, chunks, n_chunks: int, seqs, n_seqs: int, cum, dt) -> None:
        """Portions of prompts (lists as the C ABI describes them).  ``cum``: scratch, a row per token; with
        ``dt`` both are [heads, rows]."""
        a, lib = self.args, native.load()
        a.cum, a.ldcum, a.dt = cum.data_ptr(), cum.stride(0), _p(dt)
        a.chunks, a.n_chunks, a.seqs, a.n_seqs = chunks.data_ptr(), n_chunks, seqs.data_ptr(), n_seqs
        ws = recur_workspace(lib.exo_recur_workspace(C.byref(a)), chunks.device)
        check(lib.exo_recur_chunks(C.byref(a), ws.data_ptr(), ws.numel(), _stream()), "recur_chunks")


def gated_norm(y, gate, gain, out, n: int, width: int, groups: int, eps: float, gate_first: bool, sigmoid: bool = False,
               part: int | None = None, peaks=None) -> None:
    """out[:n] = RMS norm of ``groups`` equal parts of y (gain repeating with its own length), with silu(gate) -
    or ``sigmoid`` - ahead of the norm or behind it.  ``part``: columns from one part of y to the next; ``peaks``
    float32 [rows, groups]: a part is first divided by max(|the entry behind it|, exp(-peak)) + 1e-6."""
    a = native.GatedNorm(y=y.data_ptr(), gate=gate.data_ptr(), gain=gain.data_ptr(), out=out.data_ptr(), width=width,
                         groups=groups, period=gain.numel(), ldy=y.stride(0), ldg=gate.stride(0), ldo=out.stride(0),
                         gate_first=int(gate_first), dtype=_code(out), eps=eps, ldpart=part or width // groups, peaks=_p(peaks),
                         ldpeaks=0 if peaks is None else peaks.stride(0), den=width // groups, sigmoid=int(sigmoid))
    check(native.load().exo_gated_norm_rows(C.byref(a), None, n, _stream()), "gated_norm")
