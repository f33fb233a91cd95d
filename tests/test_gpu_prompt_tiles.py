"""The matrix-core GEMM's tiles for prompts, at the sizes where a tile ends: against float64 products of the
weights as the kernel forms them (scale * code + bias, rounded to bf16 once)."""

from __future__ import annotations

import math
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
if not torch.cuda.is_available():
    pytest.skip("needs a GPU", allow_module_level=True)

from exo_amd import dense_ops, native, ops  # noqa: E402
from exo_amd.ops import QuantizedWeight  # noqa: E402


def packed(N, K, bits, seed, device):
    g = torch.Generator(device=device).manual_seed(seed)
    w = torch.randint(-2**31, 2**31 - 1, (N, K * bits // 32), dtype=torch.int32, device=device, generator=g)
    top = float(2**bits - 1)
    s = (torch.rand(N, K // 64, device=device, generator=g) * 0.1 + 0.05) / top
    return QuantizedWeight(w, s.bfloat16(), (-s * top * 0.5).bfloat16(), bits)


def weights64(q: QuantizedWeight):
    codes = ops.unpack_codes(q.weight, q.bits).double().view(q.N, -1, 64)
    return (codes * q.scales.double()[..., None] + q.biases.double()[..., None]).float().bfloat16().double().view(q.N, -1)


def check(got, x, w, residual=None, what=""):
    """One bf16 rounding of the sum (and one more of the sum with the residual), float32 sums over K terms in any
    order: K * 2^-24 of the sum of their magnitudes."""
    want = x.double() @ w.T
    slack = x.shape[1] * 2.0**-24 * (x.double().abs() @ w.abs().T)
    size = want.abs()
    if residual is not None:
        want = want + residual.double()
        size = size + want.abs()
    bad = (got.double() - want).abs() > 2.0**-8 * size + slack + 1e-30
    assert not bad.any(), f"{what}: {int(bad.sum())} of {bad.numel()} outputs, first at {bad.nonzero()[0].tolist()}"


# short ranges of K, which leave prompts to the 128-row tiles: 6, 134 and 192 rows in the last 256, whole rounds and
# a nearly empty last one; ragged columns
@pytest.mark.parametrize("M,N,K,bits", [(1030, 16400, 256, 4), (1030, 16397, 512, 8), (902, 16640, 256, 4),
                                        (960, 16400, 256, 8), (2048, 8192, 256, 4), (513, 32776, 256, 4)])
def test_prompt_gemm_at_tile_edges(device, M, N, K, bits):
    q = packed(N, K, bits, M + N, device)
    g = torch.Generator(device=device).manual_seed(M)
    x = torch.randn(M, K, device=device, generator=g).bfloat16()
    r = torch.randn(M, N, device=device, generator=g).bfloat16()
    check(ops.quantized_matmul(x, q), x, weights64(q), what=f"{M}x{N}x{K}")
    check(ops.quantized_matmul(x, q, residual=r), x, weights64(q), r, what=f"{M}x{N}x{K} with residual")


@pytest.mark.parametrize("M,N,K,bits", [(1030, 8200, 256, 4), (300, 14336, 512, 8), (700, 8197, 256, 4)])
def test_prompt_pair_gemm_at_tile_edges(device, M, N, K, bits):
    """The gate and up projections in one launch have the bits of two launches and the SwiGLU kernel."""
    gate, up = packed(N, K, bits, M, device), packed(N, K, bits, N, device)
    x = torch.randn(M, K, device=device, generator=torch.Generator(device=device).manual_seed(K)).bfloat16()
    want = ops.swiglu(ops.qmm(x, gate), ops.qmm(x, up))
    assert torch.equal(ops.qmm_swiglu(x, gate, up).view(torch.int16), want.view(torch.int16))
    check(ops.qmm(x, gate), x, weights64(gate), what=f"gate {M}x{N}x{K}")


# the same edges where K is long enough for the 256 x 256 tile: two, four, six and eight blocks of 32 rows in the last
# tile of a column, a last round in halves, the second of which holds no row, ragged columns
@pytest.mark.parametrize("M,N,K,bits,pair", [(1030, 12288, 4096, 4, False), (900, 16397, 4352, 8, False), (960, 16640, 4096, 4, False), (1024, 8264, 4096, 8, False),
                                             (600, 14336, 4096, 4, True), (1000, 8200, 3072, 8, True), (300, 14330, 3328, 4, True), (513, 14336, 4352, 8, True)])
def test_large_tile_at_tile_edges(device, M, N, K, bits, pair):
    gate = packed(N, K, bits, M, device)
    x = torch.randn(M, K, device=device, generator=torch.Generator(device=device).manual_seed(K)).bfloat16()
    name = f"qmm_kernel<{bits}, 8, false, true, {str(pair).lower()}, true>"
    if pair:
        up = packed(N, K, bits, N, device)
        got = ops.qmm_swiglu(x, gate, up)
        assert native.last_variant() == name, native.last_variant()
        a, b = ops.qmm(x, gate), ops.qmm(x, up)
        check(a, x, weights64(gate), what=f"gate {M}x{N}x{K}")
        assert torch.equal(got.view(torch.int16), ops.swiglu(a, b).view(torch.int16))
        return
    r = torch.randn(M, N, device=device, generator=torch.Generator(device=device).manual_seed(M)).bfloat16()
    got = ops.quantized_matmul(x, gate)
    assert native.last_variant() == name, native.last_variant()
    check(got, x, weights64(gate), what=f"{M}x{N}x{K}")
    check(ops.quantized_matmul(x, gate, residual=r), x, weights64(gate), r, what=f"{M}x{N}x{K} with residual")


@pytest.mark.parametrize("M,N,K,bits,pair", [(4096, 5120, 2048, 4, False), (1030, 16400, 512, 4, False), (1500, 8192, 2048, 4, True), (1000, 8200, 1024, 4, True)])
def test_short_ranges_of_k_take_the_small_tile(device, M, N, K, bits, pair):
    gate = packed(N, K, bits, M, device)
    x = torch.randn(M, K, device=device, generator=torch.Generator(device=device).manual_seed(K)).bfloat16()
    got = ops.qmm_swiglu(x, gate, gate) if pair else ops.quantized_matmul(x, gate)
    assert native.last_variant() == f"qmm_kernel<{bits}, 4, false, true, {str(pair).lower()}, true>", native.last_variant()
    y = ops.qmm(x, gate)
    check(y, x, weights64(gate), what=f"{M}x{N}x{K}")
    assert torch.equal(got.view(torch.int16), (ops.swiglu(y, y) if pair else y).view(torch.int16))


@pytest.mark.parametrize("rows", [1, 32, 33, 64, 65, 96, 97, 128, 129])
@pytest.mark.parametrize("K,bits", [(256, 4), (1280, 4), (256, 8), (1536, 8)])
def test_grouped_gemm_multiplies_the_rows_of_its_tile(device, rows, K, bits):
    """Experts of 1 to 129 rows beside an empty one: a tile multiplies only the blocks of 32 rows that it has."""
    E, N = 4, 264
    qs = [packed(N, K, bits, e, device) for e in range(E)]
    q = QuantizedWeight(torch.stack([t.weight for t in qs]), torch.stack([t.scales for t in qs]),
                        torch.stack([t.biases for t in qs]), bits)
    idx = torch.cat([torch.full((rows,), 2), torch.full((40,), 0), torch.full((3,), 3)]).to(torch.int32).to(device)[:, None].contiguous()
    T = idx.shape[0]
    x = torch.randn(T, 1, K, device=device, generator=torch.Generator(device=device).manual_seed(rows)).bfloat16()
    y = ops.grouped_qmm(x, q, ops.moe_group(idx, E), 1)
    for e in (0, 2, 3):
        sel = (idx[:, 0] == e).nonzero()[:, 0]
        check(y[sel, 0], x[sel, 0], weights64(qs[e]), what=f"expert {e} of {len(sel)} rows")


@pytest.mark.parametrize("N,K,bits,lines", [
    (264, 256, 4, False), (264, 512, 4, False), (264, 768, 4, False), (264, 1280, 4, False), (264, 256, 8, False), (264, 768, 8, False),
    (5128, 256, 4, True), (5128, 512, 4, True), (9000, 768, 4, True), (3208, 4096, 4, True), (5128, 768, 8, False), (5128, 4096, 8, True)])
def test_grouped_pair_has_the_bits_of_two_products(device, N, K, bits, lines):
    """Gate and up products of experts of 1 to 300 rows in one launch, whose loop requests its codes step by step or, where the chip is full, by lines and in
    another order of tiles (one block of four steps of K, an odd and an even number of them), more row tiles than XCDs and no multiple of their number,
    against the two products."""
    counts = [1, 300, 31, 0, 33, 64, 65, 128, 96, 97, 129]
    E = len(counts)
    gate, up = (QuantizedWeight(*(torch.stack(t) for t in zip(*((q.weight, q.scales, q.biases) for q in (packed(N, K, bits, 100 * s + e, device) for e in range(E))))), bits) for s in (1, 2))
    idx = torch.cat([torch.full((n,), e) for e, n in enumerate(counts)]).to(torch.int32)
    idx = idx[torch.randperm(len(idx), generator=torch.Generator().manual_seed(K))].to(device)[:, None].contiguous()
    x = torch.randn(len(idx), 1, K, device=device, generator=torch.Generator(device=device).manual_seed(K)).bfloat16()
    ws = ops.moe_group(idx, E)
    y = ops.grouped_qmm_swiglu(x, gate, up, ws, 1)
    assert native.last_variant().endswith("by steps") != lines, native.last_variant()
    a, b = ops.grouped_qmm(x, gate, ws, 1), ops.grouped_qmm(x, up, ws, 1)
    assert bits == 8 or native.last_variant().endswith("by steps") == (N < 9000), native.last_variant()
    assert torch.equal(y.view(torch.int16), ops.swiglu(a, b).view(torch.int16))
    for e in range(E):
        sel = (idx[:, 0] == e).nonzero()[:, 0]
        one = QuantizedWeight(gate.weight[e], gate.scales[e], gate.biases[e], bits)
        if len(sel):
            check(a[sel, 0], x[sel, 0], weights64(one), what=f"expert {e} of {len(sel)} rows")


# prompts whose last key tile ends with the cache or inside it, queries that see none of a workgroup's later
# tiles (300 behind 40: the second half of a split starts past the first queries), one and several heads
# per kv head, both head sizes, a scale of either sign, scores that reach far above the first tile's
@pytest.mark.parametrize("T,past,Hq,Hkv,D,spare,scale", [
    (300, 40, 32, 8, 128, 0, 1.0), (300, 40, 4, 4, 128, 7, 1.0), (9, 0, 4, 4, 64, 0, 1.0), (33, 30, 4, 1, 128, 1, -1.0),
    (257, 61, 8, 1, 64, 0, 1.0), (130, 5, 6, 2, 128, 70, 0.3), (1000, 0, 8, 2, 128, 24, 6.0), (64, 0, 8, 8, 64, 0, 6.0),
    (2100, 100, 16, 2, 128, 0, 1.0), (520, 1000, 8, 8, 64, 3, -6.0), (128, 64, 4, 2, 64, 0, 0.0),
    # contexts of one tile, its last key the cache's last and not, and one key past it
    (64, 0, 4, 4, 128, 0, 3.0), (17, 47, 8, 2, 64, 9, 1.0), (63, 1, 4, 1, 128, 5, -2.0), (1, 0, 4, 1, 64, 0, 1.0), (65, 0, 8, 1, 64, 0, 1.0)])
def test_prompt_attention_at_tile_edges(device, T, past, Hq, Hkv, D, spare, scale):
    g = torch.Generator(device=device).manual_seed(T + past)
    B, S = 2, past + T + spare
    q = torch.randn(B * T, Hq * D, device=device, generator=g).bfloat16()
    k = torch.randn(B, Hkv, S, D, device=device, generator=g)
    k = (k * torch.linspace(0.2, 1.5, S, device=device)[:, None]).bfloat16()  # later keys score higher
    v = torch.randn(B, Hkv, S, D, device=device, generator=g).bfloat16()
    pos = torch.full((B,), past, dtype=torch.int32, device=device)
    out = torch.empty_like(q)
    sc = scale * D**-0.5
    ops.sdpa_prefill(q, k, v, pos, out, sc, B, T, Hq, Hkv, D)
    keep = torch.arange(S, device=device) <= torch.arange(T, device=device)[:, None] + past
    for b in range(B):
        for h in range(Hq):
            kk, vv = k[b, h * Hkv // Hq].double(), v[b, h * Hkv // Hq].double()
            s = ((q.view(B, T, Hq, D)[b, :, h].double() @ kk.T) * sc).masked_fill(~keep, float("-inf"))
            w = s.softmax(-1)
            want = w @ vv
            # weights and the result rounded to bf16 once each (2^-9), float32 scores and sums
            slack = 2.0**-8 * (w @ vv.abs()) + 1e-5
            bad = (out.view(B, T, Hq, D)[b, :, h].double() - want).abs() > slack + 2.0**-8 * want.abs()
            assert not bad.any(), f"sequence {b} head {h}: {int(bad.sum())} outputs, first at {bad.nonzero()[0].tolist()}"


@pytest.mark.parametrize("T,D", [(64, 64), (64, 128), (300, 64), (300, 128)])  # (300: the keys of a workgroup in two halves)
def test_prompt_attention_weighs_the_largest_score_with_one(device, T, D):
    """Two keys count, of the same value row: one in the first tile, weight 1, one in the second, weight 2^a (0 < a < 8).
    The larger one's weight is 1 by the time it is rounded to bf16, and the other's share of the sum, at most 1/2, was exact when
    it was: the result is that row.  A weight of 2^a itself is off by up to 2^-8 and the row's elements by half a step or more."""
    Hq, Hkv, past = 4, 2, 128
    g = torch.Generator(device=device).manual_seed(T)
    a = torch.rand(T, Hq, device=device, generator=g).mul(7.8).add(0.1).bfloat16()
    q = torch.zeros(T, Hq, D, device=device, dtype=torch.bfloat16)
    q[..., 0], q[..., 1] = a, 1
    k = torch.zeros(1, Hkv, past + T, D, device=device, dtype=torch.bfloat16)
    k[..., 1] = -100  # weight 2^-100
    k[:, :, 3] = 0
    k[:, :, 70, 0], k[:, :, 70, 1] = 1, 0
    row = (2 - torch.randint(1, 33, (D,), device=device, generator=g) / 128).bfloat16()  # (bf16 steps of 1/128, values near 2)
    v = row.expand(1, Hkv, past + T, D).contiguous()
    out = torch.empty(T, Hq * D, device=device, dtype=torch.bfloat16)
    ops.sdpa_prefill(q.view(T, -1), k, v, torch.tensor([past], dtype=torch.int32, device=device), out, math.log(2.0), 1, T, Hq, Hkv, D)
    bad = out.view(T, Hq, D) != row
    assert not bad.any(), f"{int(bad.any(-1).sum())} of {T * Hq} queries"


@pytest.mark.parametrize("T", [20, 300])
def test_prompt_attention_with_a_scale_of_nan_is_nan(device, T):
    g = torch.Generator(device=device).manual_seed(T)
    q, k, v = (torch.randn(1, 4, T, 64, device=device, generator=g).bfloat16() for _ in range(3))
    out = torch.zeros(T, 4 * 64, device=device, dtype=torch.bfloat16)
    pos = torch.zeros(1, dtype=torch.int32, device=device)
    ops.sdpa_prefill(q.transpose(1, 2).reshape(T, -1).contiguous(), k, v, pos, out, float("nan"), 1, T, 4, 4, 64)
    assert out.isnan().all()


# 17 to 64 rows: both sizes of the row tile, a step count below, at and above the eight waves, rows of scales that are no
# whole 16-byte pieces (K of 64, 192, 832), one to seven column tiles per workgroup, K in four parts, ragged columns; and
# where the tiles that split K are faster, those
@pytest.mark.parametrize("M,N,K,bits,variant", [
    (17, 4096, 64, 4, "qmm_short<4,one,2,1> parts=1"), (32, 264, 192, 8, "qmm_short<8,one,2,1> parts=1"), (33, 4099, 832, 4, "qmm_short<4,one,4,2> parts=1"),
    (64, 12290, 512, 4, "qmm_short<4,one,4,4> parts=1"), (61, 8200, 1024, 8, "qmm_short<8,one,4,3> parts=1"), (18, 16400, 512, 4, "qmm_short<4,one,2,7> parts=1"),
    (48, 28680, 512, 4, "qmm_kernel<4, 2, false, true, false, true>"), (63, 4096, 8192, 4, "qmm_short<4,one,4,4> parts=4"),
    (31, 1030, 14336, 8, "qmm_kernel<8, 1, false, true, false, true, true>"), (31, 2050, 14336, 8, "qmm_short<8,one,2,4> parts=4"),
    (64, 40, 8192, 4, "qmm_short<4,one,4,4> parts=4"), (40, 128, 2048, 8, "qmm_short<8,one,4,1> parts=1"),
    (20, 32, 32768, 4, "qmm_kernel<4, 1, false, true, false, true, true>")])
def test_short_prompt_gemm(device, M, N, K, bits, variant):
    q = packed(N, K, bits, M + N, device)
    g = torch.Generator(device=device).manual_seed(M)
    x = torch.randn(M, K, device=device, generator=g).bfloat16()
    r = torch.randn(M, N, device=device, generator=g).bfloat16()
    w = weights64(q)
    got = ops.quantized_matmul(x, q)
    assert native.last_variant() == variant, native.last_variant()
    check(got, x, w, what=f"{M}x{N}x{K}")
    check(ops.quantized_matmul(x, q, residual=r), x, w, r, what=f"{M}x{N}x{K} with residual")
    check(ops.qmm(x, q), x, w, what=f"{M}x{N}x{K} without workspace")


@pytest.mark.parametrize("M,N,K,bits", [(17, 40, 64, 4), (33, 4100, 832, 8), (64, 14336, 512, 4), (50, 8192, 1024, 4), (24, 2050, 2048, 8)])
def test_short_prompt_pair_gemm(device, M, N, K, bits):
    """The pair in one launch has the bits of two launches and the SwiGLU kernel."""
    gate, up = packed(N, K, bits, M, device), packed(N, K, bits, N, device)
    x = torch.randn(M, K, device=device, generator=torch.Generator(device=device).manual_seed(K)).bfloat16()
    want = ops.swiglu(ops.qmm(x, gate), ops.qmm(x, up))
    assert torch.equal(ops.qmm_swiglu(x, gate, up).view(torch.int16), want.view(torch.int16))


# where the launch would be more than one round of workgroups, or its K is long, the tiles that split K stay: both sizes of
# the row tile, with and without enough steps for the ring, more rows of weights than they take, the edges of the rule
@pytest.mark.parametrize("M,N,K,bits,variant", [
    (64, 8192, 12288, 4, "qmm_kernel<4, 2, false, true, false, true, true>"), (33, 8200, 8448, 8, "qmm_kernel<8, 2, false, true, false, true, true>"),
    (64, 32768, 768, 4, "qmm_kernel<4, 2, false, true, false, true>"), (17, 30000, 512, 8, "qmm_kernel<8, 1, false, true, false, true>"),
    (32, 4100, 28672, 4, "qmm_kernel<4, 1, false, true, false, true, true>"), (40, 1000, 33024, 4, "qmm_kernel<4, 2, false, true, false, false, true>"),
    (33, 32776, 3072, 4, "qmm_kernel<4, 2, false, true, false, false, true>"), (17, 32776, 2048, 4, "qmm_kernel<4, 2, false, true, false, false, true>"),
    (32, 32776, 3072, 4, "qmm_short<4,one,2,7>"), (64, 16384, 8192, 4, "qmm_short<4,one,4,4>"), (64, 28672, 512, 8, "qmm_short<8,one,4,7>")])
def test_short_prompts_take_the_faster_tile(device, M, N, K, bits, variant):
    q = packed(N, K, bits, M + N, device)
    x = torch.randn(M, K, device=device, generator=torch.Generator(device=device).manual_seed(M)).bfloat16()
    got = ops.quantized_matmul(x, q)
    assert native.last_variant().split(" parts")[0] == variant, native.last_variant()
    check(got, x, weights64(q), what=f"{M}x{N}x{K}")


@pytest.mark.parametrize("M,N,K,bits", [(33, 32776, 512, 4), (20, 32776, 3072, 4)])
def test_wide_pair_has_the_bits_of_two_products(device, M, N, K, bits):
    """More rows of weights than one round of workgroups holds: the pair and the products alone take the same tile."""
    gate, up = packed(N, K, bits, M, device), packed(N, K, bits, N, device)
    x = torch.randn(M, K, device=device, generator=torch.Generator(device=device).manual_seed(K)).bfloat16()
    want = ops.swiglu(ops.qmm(x, gate), ops.qmm(x, up))
    assert torch.equal(ops.qmm_swiglu(x, gate, up, split_k=False).view(torch.int16), want.view(torch.int16))


# a short launch of one round against one round, two against one, two against two; up to 8192 rows of weights; a long K
@pytest.mark.parametrize("M,N,K,bits,short", [(33, 8200, 2048, 4, True), (33, 14336, 768, 8, False), (64, 16384, 1024, 4, False),
                                              (20, 20480, 2048, 4, True), (64, 20480, 1024, 4, False), (64, 8192, 512, 4, True),
                                              (64, 1024, 12288, 4, False), (20, 1024, 12288, 4, True), (20, 8200, 32768, 4, True)])
def test_short_prompt_pair_takes_the_faster_tile(device, M, N, K, bits, short):
    gate, up = packed(N, K, bits, M, device), packed(N, K, bits, N, device)
    x = torch.randn(M, K, device=device, generator=torch.Generator(device=device).manual_seed(K)).bfloat16()
    want = ops.swiglu(ops.qmm(x, gate), ops.qmm(x, up))
    got = ops.qmm_swiglu(x, gate, up, split_k=False)
    assert native.last_variant().startswith(f"qmm_short<{bits},pair" if short else f"qmm_kernel<{bits}, 2"), native.last_variant()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    check(ops.qmm(x, gate), x, weights64(gate), what=f"gate {M}x{N}x{K}")


@pytest.mark.parametrize("M,N,K,bits", [(9, 14336, 2048, 8), (16, 14336, 1024, 8), (12, 8192, 2048, 8), (9, 40, 64, 8), (16, 2050, 832, 4)])
def test_nine_to_sixteen_rows(device, M, N, K, bits):
    """Batches of an 8-bit model past the GEMV: the pair, and its products alone."""
    gate, up = packed(N, K, bits, M, device), packed(N, K, bits, N, device)
    x = torch.randn(M, K, device=device, generator=torch.Generator(device=device).manual_seed(K)).bfloat16()
    got = ops.qmm_swiglu(x, gate, up)
    assert native.last_variant().startswith(f"qmm_short<{bits},pair,2,"), native.last_variant()
    a, b = ops.qmm(x, gate), ops.qmm(x, up)
    check(a, x, weights64(gate), what=f"gate {M}x{N}x{K}")
    assert torch.equal(got.view(torch.int16), ops.swiglu(a, b).view(torch.int16))
    r = torch.randn(M, N, device=device, generator=torch.Generator(device=device).manual_seed(N)).bfloat16()
    y = torch.empty_like(r)
    ws = ops.qmm_workspace(M, N, device)  # (the product as the engine calls it past the GEMV's rows)
    native.check(native.load().exo_qmm_ws(x.data_ptr(), gate.weight.data_ptr(), gate.scales.data_ptr(), gate.biases.data_ptr(), r.data_ptr(),
                                          y.data_ptr(), ws.data_ptr(), ws.numel(), M, N, K, bits, 64, torch.cuda.current_stream().cuda_stream), "qmm")
    check(y, x, weights64(gate), r, what=f"{M}x{N}x{K} with residual")


# rows of the short GEMM, of the 128-row and of the 256-row tile; K whose scales come one by one, and in fours
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K", [(20, 64, 64), (61, 2048, 256), (33, 12290, 832), (18, 28680, 512), (63, 4096, 8192), (100, 200, 192), (200, 264, 256), (300, 8192, 768), (1030, 12288, 4096)])
def test_products_with_unit_rows_are_the_weights(device, M, N, K, bits):
    """The operand that a kernel makes of codes is bf16(scale * code + bias) bit for bit, from subnormal scales to
    those of 2^100: products with rows of one 1 are the weights themselves."""
    g = torch.Generator(device=device).manual_seed(N + bits)
    q = packed(N, K, bits, M, device)
    e = torch.randint(-133, 100, q.scales.shape, device=device, generator=g)
    e[: N // 2] = torch.randint(-12, 2, q.scales[: N // 2].shape, device=device, generator=g)
    big = torch.ldexp(torch.rand(q.scales.shape, device=device, generator=g).double() + 0.5, e)
    s = torch.where(torch.rand(e.shape, device=device, generator=g) < 0.5, -big, big).bfloat16()
    b = (-big * 2.0 ** (bits - 1)).bfloat16()
    q = QuantizedWeight(q.weight, s, b, bits)
    at = torch.randint(0, K, (M,), device=device, generator=g)
    x = torch.zeros(M, K, device=device, dtype=torch.bfloat16)
    x[torch.arange(M, device=device), at] = 1
    # (a sum adds zeros to the weight; +0 where it is -0)
    assert torch.equal(ops.quantized_matmul(x, q).double(), weights64(q).T[at])


@pytest.mark.parametrize("M,N,K", [(20, 64, 64), (61, 2048, 256), (33, 12290, 832), (18, 28680, 512), (63, 4096, 8192), (100, 200, 192), (200, 264, 256), (300, 8192, 768), (1030, 12288, 4096)])
def test_products_with_unit_rows_under_the_largest_scales(device, M, N, K):
    """4-bit scales up to the largest bf16 holds, in some groups of some rows: the weights bit for bit, there and beside."""
    g = torch.Generator(device=device).manual_seed(N + K)
    q = packed(N, K, 4, M, device)
    rand = lambda: torch.rand(q.scales.shape, device=device, generator=g)  # noqa: E731
    e = torch.randint(-12, 2, q.scales.shape, device=device, generator=g)
    e = torch.where(rand() < 0.1, torch.randint(100, 128, e.shape, device=device, generator=g), e)
    e[:, 0][rand()[:, 0] < 0.1] = 104  # (the first that cannot be multiplied by 2^24)
    size = torch.ldexp(1 + 0.9 * rand().double(), e)
    size[e == 104] = 2.0**104
    s = torch.where(rand() < 0.5, -size, size).bfloat16()
    far = e > 123
    s[-1, -1], far[-1, -1] = 2.0**127 * 1.9921875, True
    b = torch.where(far, -s.float(), torch.where(far, 0, -s.float()) * 8).bfloat16()
    # (the farthest: codes 0 and 1, so that every weight is a number: -s and 0)
    codes = q.weight.view(N, K // 64, 8)
    w = torch.where(far[..., None], codes & 0x11111111, codes).view(N, K // 8).contiguous()
    q = QuantizedWeight(w, s, b, 4)
    at = torch.randint(0, K, (M,), device=device, generator=g)
    x = torch.zeros(M, K, device=device, dtype=torch.bfloat16)
    x[torch.arange(M, device=device), at] = 1
    want = weights64(q).T[at]
    assert bool(want.isfinite().all())
    assert torch.equal(ops.quantized_matmul(x, q).double(), want)


@pytest.mark.parametrize("M,pair", [(40, True), (100, True), (600, True), (300, False)])
def test_large_scales_of_pairs_and_experts(device, M, pair):
    """The same in the gated pair (large scales in some groups of the up matrix) and in the experts' GEMM, whose rows come by a list."""
    N, K, E, top = 512, 256, 3, 2
    g = torch.Generator(device=device).manual_seed(M)
    at = torch.randint(0, K, (M,), device=device, generator=g)
    x = torch.zeros(M, K, device=device, dtype=torch.bfloat16)
    x[torch.arange(M, device=device), at] = 1

    def large(n, seed):
        q = packed(n, K, 4, seed, device)
        some = torch.rand(q.scales.shape, device=device, generator=g) < 0.1
        return QuantizedWeight(q.weight, torch.where(some, q.scales.float() * 2.0**115, q.scales.float()).bfloat16(),
                               torch.where(some, q.biases.float() * 2.0**115, q.biases.float()).bfloat16(), 4)

    if pair:
        gate, up = packed(N, K, 4, 1, device), large(N, 2)
        assert bool((up.scales.float() > 2.0**104).any())
        got, a, u = ops.qmm_swiglu(x, gate, up), weights64(gate).T[at], weights64(up).T[at]
        torch.testing.assert_close(got.double(), a * torch.sigmoid(a) * u, rtol=2.0**-7, atol=0)
        return
    q = large(E * N, 3)
    w = weights64(q).view(E, N, K)
    experts = QuantizedWeight(q.weight.view(E, N, -1), q.scales.view(E, N, -1), q.biases.view(E, N, -1), 4)
    idx = torch.stack([torch.randperm(E, device=device, generator=g)[:top] for _ in range(M)]).int()
    got = ops.grouped_qmm(x.view(M, 1, K), experts, ops.moe_group(idx, E), top)
    assert torch.equal(got.view(M, top, N).double(), w[idx.long(), :, at[:, None]])


@pytest.mark.parametrize("M,N,K,kind", [
    (129, 40004, 64, "plain"), (257, 30004, 192, "tail"), (512, 20000, 128, "act"), (300, 13000, 128, "pair"),
    (257, 4100, 8192, "split"), (600, 3076, 6144, "split"),
])
def test_dense_wide_tiles(device, M, N, K, kind):
    """The 256 x 256 tile of the float products: one row past a tile, ragged columns, one to three steps of K, and ranges of K."""
    g = torch.Generator().manual_seed(M + N)
    x, w = torch.randn(M, K, generator=g).bfloat16(), (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16()
    bias, up = torch.randn(N, generator=g), (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16()
    xd, wd, bd, ud = x.to(device), w.to(device), bias.to(device), up.to(device)
    want = x.float() @ w.float().T
    out = torch.full((M, N), 7.0, dtype=torch.bfloat16, device=device)
    if kind == "pair":
        spec = SimpleNamespace(limit=7.0, alpha=1.702, shift=1.0, cubic=0.0)
        dense_ops.glu(xd, wd, ud, out, M, spec)
        u = (x.float() @ up.float().T).clamp(-7, 7)
        want = want.clamp(max=7) * torch.sigmoid(1.702 * want.clamp(max=7)) * (u + 1)
    elif kind == "tail":  # the last 100 columns in a float32 buffer
        t = torch.empty(M, 100, device=device)
        dense_ops.linear(xd, wd, out, M, bias=bd, tail=(t, 100))
        want = want + bias
        torch.testing.assert_close(t.cpu(), want[:, -100:], rtol=1e-5, atol=1e-5)
        assert (out[:, -100:] == 7).all()
        out, want = out[:, :-100], want[:, :-100]
    else:
        after = dense_ops.After("relu2") if kind == "act" else None
        dense_ops.linear(xd, wd, out, M, after=after)
        want = want.clamp(min=0).square() if kind == "act" else want
    assert native.last_variant().startswith("dense_gemm_wide<" + ("pair" if kind == "pair" else "single")), native.last_variant()
    assert (kind == "split") != native.last_variant().endswith("x1"), native.last_variant()
    # one rounding to bf16 of a sum of K products in float32
    torch.testing.assert_close(out.float().cpu(), want, rtol=2.0 ** -8, atol=2e-5 * K ** 0.5)


@pytest.mark.parametrize("M,N,K,columns,act,mul,f32,bias", [
    (257, 30004, 192, 0, None, True, False, True), (300, 32003, 64, 0, "gelu_tanh", True, False, False), (257, 30004, 64, 0, "gelu_tanh", False, True, True),
    (300, 32003, 64, 77, None, False, True, True),
    # ranges of K: four columns per thread add them up from 2^19 results on, a fourth of them across both outputs; one with a factor, an
    # activation or 3077 columns
    (600, 3076, 6144, 77, None, False, False, True), (600, 3076, 6144, 0, None, False, True, False), (600, 3076, 6144, 0, "relu2", True, False, True),
    (600, 3077, 6144, 77, None, False, False, True),
])
def test_dense_wide_tiles_stores(device, M, N, K, columns, act, mul, f32, bias):
    """Each form of the 256 x 256 tile's store: bias, activation, factor by row number, element type or float32, a second buffer of the
    last columns that begins anywhere."""
    g = torch.Generator(device=device).manual_seed(M + N)
    x, w, factor = (torch.randn(n, k, device=device, generator=g).bfloat16() for n, k in ((M, K), (N, K), (9, N)))
    w = (w.float() * K**-0.5).bfloat16()
    rows = torch.randint(0, 9, (M,), dtype=torch.int32, device=device, generator=g)
    b = torch.randn(N, device=device, generator=g) if bias else None
    out = torch.full((M, N), 7.0, dtype=torch.float32 if f32 else torch.bfloat16, device=device)
    last = torch.full((M, 80), 7.0, device=device)
    dense_ops.linear(x, w, out, M, bias=b, tail=(last, columns) if columns else None,
                     after=dense_ops.After(act, factor if mul else None, rows if mul else None))
    assert native.last_variant().startswith("dense_gemm_wide<single"), native.last_variant()
    assert (K == 6144) != native.last_variant().endswith("x1"), native.last_variant()
    y = x.float() @ w.float().T + (b if bias else 0)
    assert bool((out[:, N - columns:] == 7).all()) and bool((last[:, columns:] == 7).all())
    # the sum of K products and a bias in float32
    torch.testing.assert_close(last[:, :columns], y[:, N - columns:], rtol=2.0**-20, atol=2e-5)
    y = y[:, : N - columns]
    if act:
        y = torch.nn.functional.gelu(y, approximate="tanh") if act == "gelu_tanh" else y.clamp(min=0).square()
    if mul:
        y = y * factor[rows.long(), : N - columns].float()
    # one rounding to bf16 (none to float32) of sums that are off by 2e-5; squared and times a factor of up to 5, ten times that
    rtol = (0 if f32 else 2.0**-8) + 2e-5
    torch.testing.assert_close(out[:, : N - columns].float(), y, rtol=rtol, atol=2e-4)


@pytest.mark.parametrize("tail", [False, True])
@pytest.mark.parametrize("ld,wide", [(2097136, True), (2097152, False), (2200000, False)])
def test_dense_float_outputs_of_long_rows(device, ld, wide, tail):
    """Rows of a float32 output so far apart that 256 of them reach the offset of dropped stores: the 128-row tile, and nothing
    beside the ragged columns of either output is written."""
    M, N, K, T = 257, 30005, 64, 117
    g = torch.Generator().manual_seed(ld)
    x, w = torch.randn(M, K, generator=g).bfloat16(), torch.randn(N, K, generator=g).bfloat16()
    far = torch.full((M, ld), 7.0, device=device)
    if tail:  # the last columns go to the far buffer
        near = torch.full((M, N), 7.0, dtype=torch.bfloat16, device=device)
        dense_ops.linear(x.to(device), w.to(device), near, M, tail=(far, T))
        assert bool((near[:, N - T :] == 7).all())
        torch.testing.assert_close(near[:, : N - T].float().cpu(), (x.float() @ w.float().T)[:, : N - T], rtol=2.0**-8, atol=1e-5)
    else:
        T = N
        dense_ops.linear(x.to(device), w.to(device), far[:, :N], M)
    assert native.last_variant().startswith("dense_gemm_wide<" if wide else "dense_gemm<"), native.last_variant()
    torch.testing.assert_close(far[:, :T].cpu(), (x.float() @ w.float().T)[:, N - T :], rtol=1e-5, atol=1e-5)
    assert bool((far[:, T:] == 7).all())


@pytest.mark.parametrize("M,N,K,pair,wide", [(520, 40001, 960, False, False), (520, 40001, 1024, False, True), (257, 32001, 64, False, True),
                                             (520, 30002, 192, True, False), (520, 30002, 1024, True, True)])
def test_dense_wide_tiles_of_short_k(device, M, N, K, pair, wide):
    """More 256 x 256 tiles than CUs only over K of 1024 and more."""
    g = torch.Generator(device=device).manual_seed(K)
    x, w, u = ((torch.randn(n, K, device=device, generator=g) * f).bfloat16() for n, f in ((M, 1), (N, K**-0.5), (N, K**-0.5)))
    out, want = torch.empty(M, N, dtype=torch.bfloat16, device=device), x.float() @ w.float().T
    if pair:
        dense_ops.glu(x, w, u, out, M, SimpleNamespace(limit=7.0, alpha=1.702, shift=1.0, cubic=0.0))
        want = want.clamp(max=7) * torch.sigmoid(1.702 * want.clamp(max=7)) * ((x.float() @ u.float().T).clamp(-7, 7) + 1)
    else:
        dense_ops.linear(x, w, out, M)
    assert native.last_variant().startswith("dense_gemm_wide<") == wide, native.last_variant()
    # one rounding to bf16 of a sum of K products in float32
    torch.testing.assert_close(out.float(), want, rtol=2.0**-8, atol=2e-5 * K**0.5)
