"""Decode attention around the context lengths from which its keys are split over workgroups, against float64."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
if not torch.cuda.is_available():
    pytest.skip("needs a GPU", allow_module_level=True)

from exo_amd import ops  # noqa: E402


def rotated(x, pos, inv):
    a = pos.double()[:, None, None] * inv.double()
    lo, hi = x.double().chunk(2, -1)
    return torch.cat([lo * a.cos() - hi * a.sin(), hi * a.cos() + lo * a.sin()], -1).float().bfloat16().double()


# one workgroup up to 256 keys of 128, or of 64 up to 448, 384 and 256 with one, two and four heads in it (the matrix-core kernel, 16 and more pairs of 128: a tile of 32 cached keys for each of its six or eight waves), several
# beyond; lengths differ inside a batch, and a second call finds the hand-over's counters as the first left them
@pytest.mark.parametrize("Hq,Hkv,D,S,lens", [
    (32, 8, 128, 4096, [1]), (32, 8, 128, 4096, [256]), (32, 8, 128, 4096, [257]), (32, 8, 64, 600, [512]), (32, 8, 64, 600, [513]),
    (32, 8, 64, 600, [448]), (32, 8, 64, 600, [449]), (32, 8, 64, 600, [384, 385, 383, 600]), (32, 8, 64, 600, [256, 257, 255, 1, 512, 300, 64, 33]),
    (16, 16, 64, 200, [130, 1]), (64, 4, 128, 1100, [255, 1024]), (32, 8, 128, 1024, [1, 255, 256, 257, 513, 700, 129, 2]),
    (32, 4, 128, 700, [256, 257, 31, 600]), (64, 4, 128, 300, [256, 300, 128, 129])])
def test_decode_attention_around_the_first_split(device, Hq, Hkv, D, S, lens):
    g = torch.Generator(device=device).manual_seed(Hq + sum(lens))
    B = len(lens)
    kc, vc = (torch.randn(B, Hkv, S, D, device=device, generator=g).bfloat16() for _ in range(2))
    qkv = torch.randn(B, (Hq + 2 * Hkv) * D, device=device, generator=g).bfloat16()
    pos = torch.tensor(lens, dtype=torch.int32, device=device) - 1
    inv = 1e4 ** (-torch.arange(0, D, 2, dtype=torch.float32, device=device) / D)
    ws, out = ops.sdpa_decode_workspace(B, Hq, D, device), torch.empty(B, Hq * D, dtype=torch.bfloat16, device=device)
    x = qkv.view(B, Hq + 2 * Hkv, D)
    q, k = rotated(x[:, :Hq], pos, inv), rotated(x[:, Hq : Hq + Hkv], pos, inv)
    for _ in range(2):
        ops.attn_decode(qkv, kc, vc, pos, inv, out, ws, D**-0.5, B, Hq, Hkv, D, rope_tab=ops.rope_table(inv, S, D))
        for b, n in enumerate(lens):
            for h in range(Hq):
                kk = torch.cat([kc[b, h * Hkv // Hq, : n - 1].double(), k[b, h * Hkv // Hq][None]])
                vv = torch.cat([vc[b, h * Hkv // Hq, : n - 1].double(), x[b, Hq + Hkv + h * Hkv // Hq].double()[None]])
                w = ((kk @ q[b, h]) * D**-0.5).softmax(0)
                got, want = out[b].view(Hq, D)[h].double(), w @ vv
                # q and k rotated in float32 and rounded to bf16 once (a last place apart here and there: 2^-8 of a
                # score's terms), weights and result rounded to bf16
                slack = 2.0**-6 * (w @ vv.abs()) + 2.0**-8 * want.abs() + 1e-5
                assert ((got - want).abs() <= slack).all(), f"sequence {b} of {n} keys, head {h}"
        assert not ws[: 4 * B * Hkv].view(torch.int32)[: B * Hkv].any()


@pytest.mark.parametrize("B,Hq,Hkv,D,keys", [(1, 32, 8, 128, 40), (1, 32, 4, 128, 700), (8, 32, 8, 128, 700), (2, 8, 2, 64, 300), (8, 32, 4, 128, 100)])
def test_decode_attention_into_any_element(device, B, Hq, Hkv, D, keys):
    """An output that begins at an odd element of its buffer: the bits of one that does not, and nothing beside it."""
    g = torch.Generator(device=device).manual_seed(keys)
    kc, vc = (torch.randn(B, Hkv, 1024, D, device=device, generator=g).bfloat16() for _ in range(2))
    qkv = torch.randn(B, (Hq + 2 * Hkv) * D, device=device, generator=g).bfloat16()
    pos = torch.full((B,), keys - 1, dtype=torch.int32, device=device)
    inv = 1e4 ** (-torch.arange(0, D, 2, dtype=torch.float32, device=device) / D)
    ws, n = ops.sdpa_decode_workspace(B, Hq, D, device), B * Hq * D
    outs = [torch.full((n + 2,), 7.0, dtype=torch.bfloat16, device=device) for _ in range(2)]
    for at, out in enumerate(outs):
        ops.attn_decode(qkv, kc, vc, pos, inv, out[at : at + n], ws, D**-0.5, B, Hq, Hkv, D)
    assert torch.equal(outs[0][:n], outs[1][1 : n + 1]) and bool((outs[0][n:] == 7).all()) and bool((outs[1][:: n + 1] == 7).all())


# the launch is laid out for more keys than the rows hold: splits without a tile of 32 keys (four to a split) leave the
# merge to the others, down to one that writes the result itself; rows of one launch differ, a second launch
# finds the counters as the first left them
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,last,window,keep", [(700, [699, 128, 0], None, 0), (700, [127, 255, 256], None, 0), (600, [599, 300, 31], 100, 40)])
def test_paged_rows_with_idle_splits(device, dtype, T, last, window, keep):
    from exo_amd import dense_ops as D
    from exo_amd.paged_cache import PagedKVCache
    from tests import test_gpu_gekazen as G
    from tests.stack_util import TOL, close, host

    spec = G.make_spec(8, 2, 64, 64, window, keep)
    rows = torch.randn(T, (8 + 2 * 2) * 64, generator=torch.Generator().manual_seed(T)).numpy()
    cache = PagedKVCache([(2, 64, 64)], 3, 2048, "cuda", dtype)
    att = D.PagedAttention(spec, torch.tensor(spec.slopes, dtype=torch.float32, device=device), 0, cache, 1e-6)
    qkv = torch.tensor(rows, device=device).to(dtype)
    held = qkv.float().cpu().numpy().reshape(T, 12, 64)
    i32 = dict(dtype=torch.int32, device=device)
    cache.reserve([1], T)
    att.append(qkv, torch.full((T,), 1, **i32), torch.arange(T, **i32), T)
    want = G.attn_oracle(spec, (held[:, :8], held[:, 8:10], held[:, 10:]), 1e-6, dtype)
    part, out = qkv[last].contiguous(), torch.zeros(len(last), 512, dtype=dtype, device=device)
    for keys in (2000, T, 2000):
        out.zero_()
        att.rows(part, out, torch.full((len(last),), 1, **i32), torch.tensor(last, **i32), len(last), keys, append=False)
        close(host(out).reshape(len(last), 8, 64), want[last], 3 * TOL[dtype], f"{keys} keys allowed for")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("vdim,offset", [(63, 0), (1, 0), (64, 4), (33, 4)])
def test_paged_rows_merge_partials_at_any_float(device, monkeypatch, dtype, vdim, offset):
    """Several splits whose partials do not lie at multiples of eight bytes: an odd value width, a workspace four bytes further."""
    from exo_amd import dense_ops as D
    from exo_amd import native
    from exo_amd.paged_cache import PagedKVCache
    from tests import test_gpu_gekazen as G
    from tests.stack_util import TOL, close, host

    T, last, cols = 700, [699, 300, 0], 10 * 64 + 2 * vdim
    spec = G.make_spec(8, 2, 64, vdim, None, 0)
    rows = torch.randn(T, cols, generator=torch.Generator().manual_seed(vdim)).to(device).to(dtype)
    cache = PagedKVCache([(2, 64, vdim)], 3, 2048, "cuda", dtype)
    att = D.PagedAttention(spec, torch.tensor(spec.slopes, dtype=torch.float32, device=device), 0, cache, 1e-6)
    held = rows.float().cpu().numpy()
    i32 = dict(dtype=torch.int32, device=device)
    cache.reserve([1], T)
    att.append(rows, torch.full((T,), 1, **i32), torch.arange(T, **i32), T)
    q, k, v = held[:, :512].reshape(T, 8, 64), held[:, 512:640].reshape(T, 2, 64), held[:, 640:].reshape(T, 2, vdim)
    want = G.attn_oracle(spec, (q, k, v), 1e-6, dtype)
    held_ws = torch.zeros(1 << 22, dtype=torch.uint8, device=device)
    monkeypatch.setattr(D, "attn_workspace", lambda *a: held_ws[offset:])
    part, out = rows[last].contiguous(), torch.full((len(last), 8 * vdim + 1), 7.0, dtype=dtype, device=device)
    for _ in range(2):
        att.rows(part, out, torch.full((len(last),), 1, **i32), torch.tensor(last, **i32), len(last), T, append=False)
        assert "splits=1 " not in native.last_variant(), native.last_variant()
        close(host(out[:, : 8 * vdim]).reshape(len(last), 8, vdim), want[last], 3 * TOL[dtype], f"values of {vdim}")
        assert bool((out[:, 8 * vdim] == 7).all())


# single steps of queries and keys without norm or rotation: rows copied in 16 bytes (or element by element where the width is no multiple of
# that), one, two or four columns of the result to a thread, keys at either end of a tile and of a page, one workgroup and several
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(8, 1, 128, 128), (4, 1, 64, 66), (2, 2, 64, 64), (6, 2, 36, 20), (1, 1, 16, 3), (16, 1, 256, 32)])
def test_paged_rows_of_plain_queries(device, dtype, shape):
    from tests import test_gpu_gekazen as G
    from tests.stack_util import TOL, close

    spec = G.make_spec(*shape, None, 0, slopes=False, unit=False)
    cuts = [30, 1, 1, 1, 1, 29, 1, 1, 1, 61, 1, 1, 1, 126, 1, 1, 1, 1]
    rows, qkv = G.attn_case(spec, sum(cuts), seed=shape[2])
    want = G.attn_oracle(spec, qkv, 1e-6)
    close(G.run_portions(spec, rows, cuts, dtype, 1e-6), want, 3 * TOL[dtype], str(shape))


# bits of the outputs, recorded on the card: the keys of a tile meet in the sums in their order, and a change of it, which no tolerance shows, changes
# them (and with them what a decoder gives for the same request)
@pytest.mark.parametrize("heads,kv_heads,dim,keys,scale,digest", [
    (32, 4, 128, 700, 0.02, "e79732b5ac35948f"), (16, 8, 64, 48, 0.5, "ec73869fddee6247"), (8, 2, 64, 2000, 0.5, "96b7dfdbd97c0ac2")])
def test_paged_rows_keep_the_order_of_keys(device, heads, kv_heads, dim, keys, scale, digest):
    import hashlib

    from exo_amd import dense_ops as D
    from exo_amd.paged_cache import PagedKVCache
    from tests import test_gpu_gekazen as G

    spec = G.make_spec(heads, kv_heads, dim, dim, None, 0, scale=scale, slopes=False)
    cache = PagedKVCache([(kv_heads, dim, dim)], 2, keys + 64, "cuda", torch.bfloat16)
    att = D.PagedAttention(spec, None, 0, cache, 1e-6)
    qkv = torch.randn(keys, (heads + 2 * kv_heads) * dim, generator=torch.Generator().manual_seed(keys)).to(device).bfloat16()
    i32 = dict(dtype=torch.int32, device=device)
    cache.reserve([1], keys)
    att.append(qkv, torch.full((keys,), 1, **i32), torch.arange(keys, **i32), keys)
    last = torch.tensor([keys - 1, keys // 2], **i32)
    out = torch.zeros(2, heads * dim, dtype=torch.bfloat16, device=device)
    att.rows(qkv[last.long()].contiguous(), out, torch.full((2,), 1, **i32), last, 2, keys, append=False)
    got = hashlib.sha256(out.view(torch.int16).cpu().numpy().tobytes()).hexdigest()[:16]
    assert got == digest, got
