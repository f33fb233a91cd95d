"""Parity of every HIP kernel, called through the C ABI, against the CPU oracle.

Bar: bit-exact for codes / dequantised weights / indices; rtol 2e-2 (+ atol =
rtol*rms) for bf16 activations.
"""

import numpy as np
import pytest
import torch

from oracle import affine
from oracle import ops as O
from tests.util import (
    assert_close, assert_close_stat, n_bits, n_f32, rand_bf16, rand_quantized, rng, t_bf16, t_qw, t_u32,
)

pytestmark = pytest.mark.gpu

from exo_amd import native, ops  # noqa: E402


def test_library_loads_and_reports_mode():
    lib = native.load()
    assert lib.exo_abi_version() == 1
    assert lib.exo_dequant_two_roundings() in (0, 1)


@pytest.mark.parametrize("bits", [4, 8])
def test_unpack_codes_bit_exact(device, bits):
    w = rng(1).integers(0, 2**32, size=(37, 96), dtype=np.uint64).astype(np.uint32)
    got = ops.unpack_codes(t_u32(w, device), bits).cpu().numpy()
    np.testing.assert_array_equal(got, affine.unpack_codes(w, bits))


@pytest.mark.parametrize("bits", [4, 8])
def test_dequantize_bit_exact(device, bits):
    trip = rand_quantized(50, 512, bits, seed=3)
    got = n_bits(ops.dequantize(t_qw(trip, bits, device)))
    mode = "M1" if native.load().exo_dequant_two_roundings() else "M2"
    want = affine.dequantize(*trip, 64, bits, mode)
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("bits", [4, 8])
def test_dequantize_all_codes_extreme_scales(device, bits):
    # every code value at every slot, with scales/biases spanning magnitudes
    K = 256 if bits == 8 else 64
    per = 1 << bits
    codes = (np.arange(per * K).reshape(per, K) // 1 + np.arange(per)[:, None]) % per
    codes = np.tile(codes.astype(np.uint8), (1, 1))
    w = affine.pack_codes(codes, bits)
    G = K // 64
    s = affine.f32_to_bf16_bits((rng(5).standard_normal((per, G)) * 10.0 ** rng(6).integers(-6, 3, (per, G))).astype(np.float32))
    b = affine.f32_to_bf16_bits((rng(7).standard_normal((per, G)) * 10.0 ** rng(8).integers(-6, 3, (per, G))).astype(np.float32))
    got = n_bits(ops.dequantize(t_qw((w, s, b), bits, device)))
    mode = "M1" if native.load().exo_dequant_two_roundings() else "M2"
    np.testing.assert_array_equal(got, affine.dequantize(w, s, b, 64, bits, mode))


@pytest.mark.parametrize("bits", [4, 8])
def test_embed_bit_exact(device, bits):
    trip = rand_quantized(300, 256, bits, seed=9)
    ids = np.array([0, 299, 5, 5, 17, 128], np.int32)
    got = n_bits(ops.embed(torch.from_numpy(ids).to(device), t_qw(trip, bits, device)))
    mode = "M1" if native.load().exo_dequant_two_roundings() else "M2"
    want = affine.dequantize(trip[0][ids], trip[1][ids], trip[2][ids], 64, bits, mode)
    np.testing.assert_array_equal(got, want)


QMV_SHAPES = [  # (N, K)
    (256, 4096), (64, 2048), (128, 14336), (96, 768), (64, 1536), (200, 8192), (128, 64),
    (72, 192), (160, 7168),
]


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("N,K", QMV_SHAPES)
@pytest.mark.parametrize("M", [1, 2, 3, 7, 16])
def test_qmv(device, bits, N, K, M):
    trip = rand_quantized(N, K, bits, seed=N + K + bits)
    x = rand_bf16((M, K), seed=M + K)
    got = n_f32(ops.quantized_matmul(t_bf16(x, device), t_qw(trip, bits, device)))
    want = affine.qmm(x, *trip, 64, bits)
    assert_close(got, want, what=f"qmv {M}x{N}x{K} b{bits}")


@pytest.mark.parametrize("bits", [4, 8])
def test_qmv_is_accurate_beyond_bf16(device, bits):
    # float32 accumulation: before the final rounding the result should sit within
    # about one bf16 ulp of the float64 value.
    N, K, M = 512, 4096, 1
    trip = rand_quantized(N, K, bits, seed=77)
    x = rand_bf16((M, K), seed=78)
    got = n_f32(ops.quantized_matmul(t_bf16(x, device), t_qw(trip, bits, device)))
    wd = affine.dequantize_f32(*trip, 64, bits).astype(np.float64)
    exact = x.astype(np.float64) @ wd.T
    err = np.abs(got - exact)
    assert np.all(err <= np.abs(exact) * 2.0**-8 + 1e-4), err.max()


@pytest.mark.parametrize("bits", [4, 8])
def test_qmv_residual(device, bits):
    N, K, M = 192, 2048, 3
    trip = rand_quantized(N, K, bits, seed=21)
    x = rand_bf16((M, K), seed=22)
    r = rand_bf16((M, N), seed=23)
    got = n_f32(ops.quantized_matmul(t_bf16(x, device), t_qw(trip, bits, device), residual=t_bf16(r, device)))
    want = affine.bf16_round(affine.qmm(x, *trip, 64, bits) + r)
    assert_close(got, want, what="qmv+residual")


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M", [1, 2, 4, 9, 16])
def test_qmv_swiglu(device, bits, M):
    N, K = 320, 2048
    g = rand_quantized(N, K, bits, seed=31)
    u = rand_quantized(N, K, bits, seed=32)
    x = rand_bf16((M, K), seed=33)
    got = n_f32(ops.qmv_swiglu(t_bf16(x, device), t_qw(g, bits, device), t_qw(u, bits, device)))
    want = O.swiglu(affine.qmm(x, *g, 64, bits), affine.qmm(x, *u, 64, bits))
    assert_close(got, want, what="qmv_swiglu")


W16_SHAPES = [  # (N, K): rows of 6 | 8 | 14 | 16 waves x 1 | 2 slices, K split 2 | 4 ways
    (4112, 768), (2064, 1024), (1008, 2560), (1040, 3584), (528, 4096), (272, 8192), (304, 14336),
]


@pytest.mark.parametrize("N,K", W16_SHAPES)
@pytest.mark.parametrize("M", [5, 8, 11, 16])
def test_qmv_16x16x32_kernel_shapes(device, N, K, M):
    """The 16x16x32 matrix-core GEMV (4-bit, 5..16 rows) over its wave /
    slice layouts: plain, with residual, with the fused RMSNorm (rows of up to 4096 elements),
    and the (gate, up) pair with SwiGLU; every result against the oracle, every launch asserted
    to have reached that kernel."""
    bits = 4
    trip = rand_quantized(N, K, bits, seed=N + K)
    qw = t_qw(trip, bits, device)
    x = rand_bf16((M, K), seed=M + K, scale=1.5)
    xt = t_bf16(x, device)
    want = affine.qmm(x, *trip, 64, bits)
    got = ops.quantized_matmul(xt, qw)
    assert native.last_variant().startswith("qmv_w16<1,"), native.last_variant()
    if K > 4096:
        assert "kparts=1" not in native.last_variant(), native.last_variant()
    assert_close(n_f32(got), want, what=f"w16 {M}x{N}x{K}")
    r = rand_bf16((M, N), seed=N + 3)
    got = ops.quantized_matmul(xt, qw, residual=t_bf16(r, device))
    assert native.last_variant().startswith("qmv_w16<1,"), native.last_variant()
    assert_close(n_f32(got), affine.bf16_round(affine.bf16_round(want) + r), what=f"w16 residual {M}x{N}x{K}")
    # the split-K workspace is left clean: the same launch again gives the same bits
    again = ops.quantized_matmul(xt, qw, residual=t_bf16(r, device))
    assert torch.equal(got.view(torch.int16), again.view(torch.int16))
    if K <= 4096:
        w = affine.bf16_round(rand_bf16((K,), seed=6) * 0.1 + 1.0)
        xn = O.rms_norm(x, w, 1e-5)
        got = ops.quantized_matmul(xt, qw, norm_weight=t_bf16(w, device), eps=1e-5)
        assert native.last_variant().startswith("qmv_w16<1,") and "norm" in native.last_variant(), native.last_variant()
        assert_close(n_f32(got), affine.qmm(xn, *trip, 64, bits), what=f"w16 norm {M}x{N}x{K}")
        up = rand_quantized(N, K, bits, seed=N + K + 1)
        got = ops.qmv_swiglu(xt, qw, t_qw(up, bits, device), norm_weight=t_bf16(w, device), eps=1e-5)
        assert native.last_variant().startswith("qmv_w16<2,"), native.last_variant()
        assert_close(n_f32(got), O.swiglu(affine.qmm(xn, *trip, 64, bits), affine.qmm(xn, *up, 64, bits)),
                     what=f"w16 pair {M}x{N}x{K}")


def most_of_group(xa):
    """The largest of each element's quantisation group."""
    return xa.view(xa.shape[0], -1, 64).amax(2).repeat_interleave(64, 1)


@pytest.mark.parametrize("bits,N,K,pair,plain", [
    (4, 4099, 2048, False, False), (4, 16389, 2048, False, True), (4, 2050, 4096, False, False), (4, 4301, 4096, False, True), (4, 1371, 6144, False, False),
    (4, 2611, 6144, False, True), (4, 1030, 8192, False, False), (4, 1957, 8192, False, True),
    (8, 2049, 2048, False, False), (8, 8195, 2048, False, True), (8, 1025, 4096, False, False), (8, 2001, 4096, False, True), (8, 687, 6144, False, False),
    (8, 1307, 6144, False, True), (8, 521, 8192, False, False), (8, 979, 8192, False, True),
    (4, 2051, 2048, True, False), (4, 8193, 2048, True, True), (4, 689, 6144, True, False), (4, 1307, 6144, True, True), (4, 514, 8192, True, False), (4, 979, 8192, True, True),
    (8, 1027, 2048, True, False), (8, 2151, 2048, True, True), (8, 4097, 4096, True, True), (8, 653, 6144, True, True), (8, 259, 8192, True, False), (8, 491, 8192, True, True),
])
def test_qmv_planes(device, bits, N, K, pair, plain):
    """One row on the integer matrix cores: last tiles of a few rows, one and several tiles per workgroup, every K, behind a norm and (launches that
    are large enough for it) without one, with a residual and without; elements of one size, a few far larger, sizes spread over many
    binades, zeros, the smallest and the largest whose results the type holds, and scales of 2^104."""
    g = torch.Generator(device=device).manual_seed(N + K)

    def rows():
        w = torch.randint(-2**31, 2**31 - 1, (N, K * bits // 32), dtype=torch.int32, device=device, generator=g)
        s, b = (torch.randn(N, K // 64, device=device, generator=g).bfloat16() * f for f in (0.02, 0.1))
        return ops.QuantizedWeight(w, s, b, bits)

    def product(x, q):
        """In float64, and how far the kernel may be off: whole-number sums are exact but for an element's last bits, 2^-30 of the
        largest of its group; a group's sum is rounded three times and K / 64 of them are added; the rounding to bf16."""
        s, b = q.scales.double()[..., None], q.biases.double()[..., None]
        codes = ops.unpack_codes(q.weight, bits).double().view(N, -1, 64)
        w = (codes * s + b).view(N, K)
        size = ((codes + 128 * (bits == 8)) * s.abs() + b.abs()).view(N, K)
        y, xa = x.double() @ w.T, x.double().abs()
        return y, 2.0**-8 * y.abs() + ((4 + K // 64) * 2.0**-24 * xa + 2.0**-30 * most_of_group(xa)) @ size.T

    q = rows()
    up = rows() if pair else None
    nw = (torch.randn(K, device=device, generator=g) * 0.1 + 1).bfloat16()
    res = torch.randn(1, N, device=device, generator=g).bfloat16()
    normal = torch.randn(1, K, device=device, generator=g)
    few, spread = normal.clone(), normal * torch.exp(4 * torch.randn(1, K, device=device, generator=g))
    few[0, ::977] *= 300
    ends = (2.0**-45, 2.0**45) if pair else (2.0**-115, 2.0**110)  # (of a pair the product of two sums)
    inputs = [("normal", normal, True, True), ("few", few, True, False)]
    if plain:
        inputs += [("normal", normal, False, True), ("few", few, False, False), ("spread", spread, False, True), ("zero", normal * 0, False, False),
                   ("small", normal * ends[0], False, False), ("large", normal * ends[1], False, False)]
    for what, x, norm, residual in inputs:
        x = x.bfloat16()
        xn = ops.rms_norm(x, nw, 1e-5) if norm else x  # (its sum of squares is in another order: a rounding of an element may differ)
        kw = dict(norm_weight=nw, eps=1e-5) if norm else {}
        y, slack = product(xn, q)
        slack = slack + (2.0**-7 * y.pow(2).mean().sqrt() if norm else 0.0)
        if pair:
            got = ops.qmv_swiglu(x, q, up, **kw)
            yu, slack_u = product(xn, up)
            slack_u = slack_u + (2.0**-7 * yu.pow(2).mean().sqrt() if norm else 0.0)
            y, slack = y * torch.sigmoid(y) * yu, (1.1 * slack + 2.0**-8 * y.abs()) * yu.abs() + y.abs() * (slack_u + 2.0**-8 * yu.abs()) + 1.1 * slack * slack_u + 1e-30
        elif residual:
            got = ops.quantized_matmul(x, q, residual=res, **kw)
            y, slack = y + res.double(), slack + 2.0**-8 * (y.abs() + res.double().abs())
        else:
            got = ops.quantized_matmul(x, q, **kw)
        assert native.last_variant().startswith("qmv_planes<%d,%d,%d," % (bits, 1 + pair, K // 2048)), native.last_variant()
        off = (got.double() - y).abs() - slack
        assert off.max() <= 0, (what, norm, off.max(), off.argmax())
    if bits == 4 and not pair:  # sums that fit the type under scales that leave no room
        big = ops.QuantizedWeight(q.weight, (q.scales.float() * 2.0**110).bfloat16(), (q.biases.float() * 2.0**110).bfloat16(), bits)
        x = normal.bfloat16()
        got = ops.quantized_matmul(x, big, norm_weight=nw, eps=1e-5)
        assert native.last_variant().startswith("qmv_planes<")
        y, slack = product(ops.rms_norm(x, nw, 1e-5), big)
        assert ((got.double() - y).abs() <= slack + 2.0**-7 * y.pow(2).mean().sqrt()).all()
    for bad in (float("inf"), float("nan")):  # reach every output, whichever wave holds them
        for at in (0, K // 2, K - 1):
            x = normal.bfloat16()
            x[0, at] = bad
            got = ops.qmv_swiglu(x, q, up, norm_weight=nw) if pair else ops.quantized_matmul(x, q, norm_weight=nw)
            assert got.isnan().all()


@pytest.mark.parametrize("bits,M,N,K,pair,norm", [
    (8, 3, 1537, 2048, False, False), (8, 2, 4100, 2048, False, True), (8, 8, 36865, 2048, False, True), (8, 5, 1, 2048, True, True), (8, 7, 17, 4096, True, False),
    (8, 6, 4113, 4096, False, True), (8, 4, 2577, 4096, False, False), (8, 3, 9, 6144, True, True), (8, 2, 35, 8192, False, True), (8, 4, 8200, 4096, True, True),
    (4, 3, 7, 2048, True, False), (4, 2, 1031, 2048, True, False), (4, 3, 2055, 2048, True, True), (4, 4, 4609, 2048, False, True), (4, 2, 33000, 2048, False, True),
    (4, 4, 2100, 4096, True, True), (4, 3, 28677, 8192, False, False), (4, 4, 14341, 8192, True, True),
])
def test_qmv_planes_rows(device, bits, M, N, K, pair, norm):
    """Two to eight rows on the integer matrix cores: last tiles of a few weight rows, one and several tiles per workgroup, one and two operands
    of rows, every K; rows of very different sizes, one of zeros, one with an element that is not a number."""
    g = torch.Generator(device=device).manual_seed(N + K + M)

    def rows():
        w = torch.randint(-2**31, 2**31 - 1, (N, K * bits // 32), dtype=torch.int32, device=device, generator=g)
        s, b = (torch.randn(N, K // 64, device=device, generator=g).bfloat16() * f for f in (0.02, 0.1))
        return ops.QuantizedWeight(w, s, b, bits)

    def product(x, q):
        """As above."""
        s, b = q.scales.double()[..., None], q.biases.double()[..., None]
        codes = ops.unpack_codes(q.weight, bits).double().view(N, -1, 64)
        y, xa = x.double() @ (codes * s + b).view(N, K).T, x.double().abs()
        size = ((codes + 128 * (bits == 8)) * s.abs() + b.abs()).view(N, K)
        return y, 2.0**-8 * y.abs() + ((4 + K // 64) * 2.0**-24 * xa + 2.0**-30 * most_of_group(xa)) @ size.T

    q, up = rows(), rows() if pair else None
    nw = (torch.randn(K, device=device, generator=g) * 0.1 + 1).bfloat16()
    res = torch.randn(M, N, device=device, generator=g).bfloat16()
    x = torch.randn(M, K, device=device, generator=g) * 2.0 ** torch.arange(0, 5 * M, 5, device=device)[:, None]
    x[:, K // 2 :] *= 2.0**-9
    if not norm:
        x[M // 2] = 0
    x = x.bfloat16()
    xn = ops.rms_norm(x, nw, 1e-5) if norm else x  # (its sum of squares is in another order: a rounding of an element may differ)
    kw = dict(norm_weight=nw, eps=1e-5) if norm else {}
    run = lambda x: ops.qmv_swiglu(x, q, up, **kw) if pair else ops.quantized_matmul(x, q, residual=res, **kw)  # noqa: E731
    got = run(x)
    assert native.last_variant().startswith(f"qmv_planes_rows<{bits},{1 + pair},{K // 2048},{4 if M <= 4 else 8}>"), native.last_variant()
    y, slack = product(xn, q)
    row_rms = lambda v: v.pow(2).mean(1, keepdim=True).sqrt()  # noqa: E731
    if norm:
        slack = slack + 2.0**-7 * row_rms(y)
    if pair:
        yu, slack_u = product(xn, up)
        if norm:
            slack_u = slack_u + 2.0**-7 * row_rms(yu)
        unit = y * torch.sigmoid(y)
        y, slack = unit * yu, (1.1 * slack + 2.0**-8 * unit.abs()) * yu.abs() + unit.abs() * (slack_u + 2.0**-8 * yu.abs()) + 1.1 * slack * slack_u + 2.0**-8 * (unit * yu).abs() + 1e-30
    else:
        y, slack = y + res.double(), slack + 2.0**-8 * (y.abs() + res.double().abs())
    assert bool(((got.double() - y).abs() <= slack).all()), float(((got.double() - y).abs() - slack).max())
    bad = x.clone()
    bad[M - 1, K - 1] = float("nan")
    other = run(bad)
    assert bool(other[M - 1].isnan().all()) and torch.equal(other[: M - 1], got[: M - 1])


@pytest.mark.parametrize("M,N,K,pair,grid", [
    (4, 976, 8192, False, 122), (3, 4464, 8192, False, 256), (8, 4112, 4096, False, 256), (2, 2053, 2048, True, 256), (5, 509, 4096, True, 128), (6, 521, 2048, False, 66), (3, 4096, 4096, False, 256),
])
def test_planes_rows_tiles_of_fewer_rows(device, M, N, K, pair, grid):
    """8 bits, fewer tiles than CUs or unequal shares of them: tiles of fewer than 16 rows (a pair: 8 of each matrix), a last tile of a part of those, and equal shares."""
    g = torch.Generator(device=device).manual_seed(N + K + M)
    ws = [ops.QuantizedWeight(torch.randint(-2**31, 2**31 - 1, (N, K // 4), dtype=torch.int32, device=device, generator=g),
                              *((torch.randn(N, K // 64, device=device, generator=g) * f).bfloat16() for f in (0.002, 0.1)), 8) for _ in range(1 + pair)]
    x, nw = torch.randn(M, K, device=device, generator=g).bfloat16(), torch.ones(K, dtype=torch.bfloat16, device=device)
    if pair:
        got = ops.qmv_swiglu(x, *ws)
    else:
        got = ops.quantized_matmul(x, ws[0], norm_weight=nw if M in (3, 4) else None, eps=1e-5)
    assert native.last_variant() == f"qmv_planes_rows<8,{1 + pair},{K // 2048},{4 if M <= 4 else 8}> grid={grid}", native.last_variant()
    xn = ops.rms_norm(x, nw, 1e-5).double() if not pair and M in (3, 4) else x.double()
    sums = []
    for q in ws:
        codes, s, b = ops.unpack_codes(q.weight, 8).double().view(N, -1, 64), q.scales.double()[..., None], q.biases.double()[..., None]
        size = xn.abs() @ ((codes + 128) * s.abs() + b.abs()).view(N, K).T
        # (a sum of K / 64 groups in float32, elements to 2^-30 of their group's largest, the norm's rounding of an element, one to bf16)
        y = xn @ (codes * s + b).view(N, K).T
        sums.append((y, ((4 + K // 64) * 2.0**-24 + 2.0**-26) * size + (2.0**-7 * y.pow(2).mean(1, keepdim=True).sqrt() if not pair else 0) + 2.0**-8 * y.abs()))
    y, slack = sums[0]
    if pair:
        (yu, slack_u), unit = sums[1], y * torch.sigmoid(y)
        y, slack = unit * yu, 1.1 * slack * (yu.abs() + slack_u) + unit.abs() * slack_u + 2.0**-8 * ((unit * yu).abs() + unit.abs() * yu.abs())
    assert bool(((got.double() - y).abs() <= slack + 1e-30).all()), float(((got.double() - y).abs() - slack).max())


@pytest.mark.parametrize("bits,M,N,K,down", [(4, 1, 8600, 2048, 0), (4, 1, 1960, 8192, 0), (8, 1, 4300, 2048, 0), (8, 1, 1400, 6144, 0), (8, 3, 1600, 2048, 0),
                                             (8, 8, 4100, 4096, 0), (4, 3, 28700, 8192, 0), (4, 1, 77, 1536, 8), (8, 2, 50, 768, 2)])
@pytest.mark.parametrize("far", [2.0**40, 2.0**-90])
def test_qmv_planes_of_far_elements(device, bits, M, N, K, down, far):
    """An element far larger than all others that meets zero weights, and elements far smaller than that one's type could hold beside
    it: the other groups' products are what they are without it."""
    g = torch.Generator(device=device).manual_seed(N + K)
    w = torch.randint(-2**31, 2**31 - 1, (N, K * bits // 32), dtype=torch.int32, device=device, generator=g)
    s, b = (torch.randn(N, K // 64, device=device, generator=g).bfloat16() * f for f in (0.02, 0.1))
    s[:, 3], b[:, 3] = 0, 0
    x = torch.randn(M, K, device=device, generator=g) * min(far, 1)
    x[:, 3 * 64 + 5] = max(far, 1)
    x = x.bfloat16()
    codes = ops.unpack_codes(w, bits).double().view(N, -1, 64)
    others = x.double()
    others[:, 3 * 64 : 4 * 64] = 0
    y = others @ (codes * s.double()[..., None] + b.double()[..., None]).view(N, K).T
    size = ((codes + 128 * (bits == 8)) * s.double().abs()[..., None] + b.double().abs()[..., None]).view(N, K)
    # (rounding to bf16; a group's sum is rounded three times, and K / 64 of them are added; elements to 2^-30 of their group's largest)
    slack = 2.0**-8 * y.abs() + ((4 + K // 64) * 2.0**-24 * others.abs() + 2.0**-30 * most_of_group(others.abs())) @ size.T
    if down:  # every slot the same row of x and expert, all but the first with no weight
        one = lambda t: t[None].contiguous()  # noqa: E731
        scores = torch.zeros(M, down, dtype=torch.bfloat16, device=device)
        scores[:, 0] = 1
        got = ops.gather_qmv_combine(x[:, None].repeat(1, down, 1), ops.QuantizedWeight(one(w), one(s), one(b), bits), torch.zeros(M, down, dtype=torch.int32, device=device),
                                     scores, scratch=torch.empty(M, down, N, dtype=torch.bfloat16, device=device))
    else:
        got = ops.quantized_matmul(x, ops.QuantizedWeight(w, s, b, bits))
    assert "planes" in native.last_variant(), native.last_variant()
    assert bool(((got.double() - y).abs() <= slack).all()), float(((got.double() - y).abs() - slack).max())


@pytest.mark.parametrize("bits,E,N,K,T,topk", [(4, 16, 5, 2048, 1, 8), (4, 8, 772, 2048, 5, 2), (8, 8, 9, 4096, 3, 4), (4, 4, 130, 8192, 2, 3), (8, 4, 66, 6144, 2, 2),
                                                   (4, 8, 24, 2048, 12, 4), (8, 4, 9, 4096, 6, 2), (8, 4, 9, 4096, 5, 2), (4, 2, 30, 4096, 6, 2), (4, 2, 30, 4096, 5, 2)])
def test_qmv_planes_of_experts(device, bits, E, N, K, T, topk):
    """The routed pair on the integer matrix cores: each (token, slot) has the outputs of its expert's own launch or, where that is
    too small for it, those of the dot products to the last place or so; just below and at the pairs an expert from which K = 4096 stays with
    the dot products."""
    g = torch.Generator(device=device).manual_seed(E + N)

    def experts():
        w = torch.randint(-2**31, 2**31 - 1, (E, N, K * bits // 32), dtype=torch.int32, device=device, generator=g)
        s, b = (torch.randn(E, N, K // 64, device=device, generator=g).bfloat16() * f for f in (0.02, 0.1))
        return ops.QuantizedWeight(w, s, b, bits)

    gate, up = experts(), experts()
    x = torch.randn(T, K, device=device, generator=g).bfloat16()
    nw = (torch.randn(K, device=device, generator=g) * 0.1 + 1).bfloat16()
    idx = torch.stack([torch.randperm(E, generator=torch.Generator().manual_seed(t))[:topk] for t in range(T)]).int().to(device)
    got = ops.gather_qmv_swiglu(x, gate, up, idx, norm_weight=nw, eps=1e-5)
    dots = K == 4096 and T * topk >= (3 if bits == 8 else 6) * E
    assert native.last_variant().startswith("qmv_rows<" if dots else "qmv_planes<"), native.last_variant()
    one = lambda q, e: ops.QuantizedWeight(q.weight[e].contiguous(), q.scales[e].contiguous(), q.biases[e].contiguous(), bits)  # noqa: E731
    for t in range(T):
        for k in range(topk):
            e = int(idx[t, k])
            want = ops.qmv_swiglu(x[t : t + 1], one(gate, e), one(up, e), norm_weight=nw, eps=1e-5)
            assert_close(n_f32(got[t, k]), n_f32(want[0]), what=f"token {t} slot {k}")


@pytest.mark.parametrize("N,K,blocks", [
    (16, 1024, 1), (8208, 768, 3), (8176, 1152, 2), (69648, 512, 9),  # one block; shares of 2 and 3; of 1 and 2; two rounds
])
@pytest.mark.parametrize("M", [6, 8, 9])
def test_qmv_16x16x32_shares_of_blocks(device, N, K, blocks, M):
    """The 16x16x32 GEMV where its workgroups' shares of row blocks differ, at both operand layouts (to 8 rows, beyond)
    and with scales in pieces of eight groups and of two."""
    trip = rand_quantized(N, K, 4, seed=N + K)
    x, r = rand_bf16((M, K), seed=M, scale=1.5), rand_bf16((M, N), seed=N)
    got = ops.quantized_matmul(t_bf16(x, device), t_qw(trip, 4, device), residual=t_bf16(r, device))
    assert native.last_variant().startswith("qmv_w16<1,1,") and f" blocks={blocks} " in native.last_variant(), native.last_variant()
    want = affine.bf16_round(affine.bf16_round(affine.qmm(x, *trip, 64, 4)) + r)
    assert_close(n_f32(got), want, what=f"w16 {M}x{N}x{K}")


@pytest.mark.parametrize("M,N,K,pair,blocks", [
    (8, 9216, 2304, False, 3), (16, 9216, 2304, True, 5), (16, 24592, 896, False, 7), (6, 40976, 2304, False, 11), (8, 36880, 2304, True, 19),
    (16, 69648, 1152, False, 6), (8, 40016, 640, False, 5), (4, 2064, 1920, False, 1), (9, 5136, 640, True, 3),
])
def test_qmv_16x16x32_rows_of_broken_pieces(device, M, N, K, pair, blocks):
    """K that is no multiple of 512: pieces of eight scales that begin in one row and end in the next, more of them than threads,
    of a matrix that begins anywhere in another; a workgroup's share is what it is for whole pieces."""
    g = torch.Generator(device=device).manual_seed(N + M)

    def rows():
        w = torch.randint(-2**31, 2**31 - 1, (N + 1, K // 8), dtype=torch.int32, device=device, generator=g)
        s, b = (torch.randn(N + 1, K // 64, device=device, generator=g).bfloat16() * f for f in (0.02, 0.1))
        return ops.QuantizedWeight(w[1:], s[1:], b[1:], 4)

    def product(q):
        """In float64, and how far a kernel may be off: sums over a slice's 128 and over the slices of |x| (|128 + code| |s| + |b|) in
        float32, and the rounding to bf16."""
        s, b = q.scales.double()[..., None], q.biases.double()[..., None]
        w = (ops.unpack_codes(q.weight, 4).double().view(N, -1, 64) * s + b).view(N, K)
        size = (143 * s.abs() + b.abs()).expand(N, K // 64, 64).reshape(N, K)
        y = x.double() @ w.T
        return y, 2.0**-8 * y.abs() + (128 + K // 64) * 2.0**-24 * (x.double().abs() @ size.T)

    x = torch.randn(M, K, device=device, generator=g).bfloat16()
    q = rows()
    want, slack = product(q)
    if pair:  # (the gate's unit grows by at most 1.1 of what the gate does)
        up = rows()
        got, (u, slack_u) = ops.qmv_swiglu(x, q, up), product(up)
        unit = want * torch.sigmoid(want)
        want, slack = unit * u, 1.1 * slack * (u.abs() + slack_u) + unit.abs() * slack_u + 2.0**-8 * (unit * u).abs()
    else:
        got = ops.quantized_matmul(x, q)
    assert native.last_variant().startswith("qmv_w16<") and f" blocks={blocks} " in native.last_variant(), native.last_variant()
    assert bool(((got.double() - want).abs() <= slack).all()), float(((got.double() - want).abs() - slack).max())


@pytest.mark.parametrize("M,N,K,per_million", [(2, 4096, 4096, 600), (4, 14336, 4096, 600), (5, 14336, 4096, 1150), (8, 14336, 4096, 1150), (8, 14336, 8192, 1150)])
def test_qmv_16x16x32_offset_leaves_no_error(device, M, N, K, per_million):
    """Outputs that are not the exact result's rounding to bf16: a share that grows with the error of the float32 sums.  With the offset
    of the codes taken out where the products are summed 115 to 155 (16 + code, up to four rows) and 580 to 755 (128 + code, up to eight) in a
    million, 1590 to 1730 with it taken out of scaled sums afterwards; the 4x4x4 kernel of up to four rows 410 to 490.  The bounds
    lie half way between, over 13 deviations of the count away from 1590 at the largest and 4 at the smallest of these shapes."""
    g = torch.Generator(device=device).manual_seed(M)
    w = torch.randn(N, K // 64, 64, device=device, generator=g) * 0.02
    lo = w.amin(-1)
    s, b = ((w.amax(-1) - lo) / 15).bfloat16(), lo.bfloat16()
    codes = ((w - b.float()[..., None]) / s.float()[..., None]).round().clamp(0, 15).int()
    packed = (codes.view(N, K // 8, 8) << torch.arange(0, 32, 4, dtype=torch.int32, device=device)).sum(-1, dtype=torch.int32)
    x = torch.randn(M, K, device=device, generator=g).bfloat16()
    got = ops.quantized_matmul(x, ops.QuantizedWeight(packed, s, b, 4))
    if M >= 4:
        assert native.last_variant().startswith("qmv_w16<"), native.last_variant()
    want = x.double() @ (codes.double() * s.double()[..., None] + b.double()[..., None]).view(N, K).T
    wrong = int((got != want.float().bfloat16()).sum())
    assert wrong * 10**6 <= per_million * M * N, wrong / (M * N)


@pytest.mark.parametrize("M,N,K,norm,pair,w16", [
    (2, 1024, 768, False, False, True), (2, 1024, 1152, True, False, False), (2, 2048, 2048, True, False, True),
    (2, 2048, 2048, False, False, False), (2, 2048, 2560, True, True, True), (3, 4096, 2048, False, False, True),
    (3, 2064, 1536, True, True, True), (4, 2048, 4096, False, False, True), (4, 2048, 8192, False, False, False),
    (4, 1040, 1024, True, True, True), (4, 2048, 2048, True, True, False), (3, 4096, 4096, False, False, True), (3, 4112, 4096, False, False, False),
    (4, 4112, 2048, False, False, False), (4, 6144, 2048, False, False, True), (3, 16400, 2560, True, True, False),
])
def test_qmv_few_rows_routes(device, M, N, K, norm, pair, w16):
    """2..4 rows on both sides of the line between the 16x16x32 and the 4x4x4 kernel."""
    trip, up = rand_quantized(N, K, 4, seed=N + K), rand_quantized(N, K, 4, seed=N + K + 1)
    x, g = rand_bf16((M, K), seed=M + K, scale=1.5), affine.bf16_round(rand_bf16((K,), seed=6) * 0.1 + 1.0)
    xn = O.rms_norm(x, g, 1e-5) if norm else x
    kw = dict(norm_weight=t_bf16(g, device), eps=1e-5) if norm else {}
    want = affine.qmm(xn, *trip, 64, 4)
    if pair:
        got = ops.qmv_swiglu(t_bf16(x, device), t_qw(trip, 4, device), t_qw(up, 4, device), **kw)
        want = O.swiglu(want, affine.qmm(xn, *up, 64, 4))
    else:
        r = rand_bf16((M, N), seed=N)
        got = ops.quantized_matmul(t_bf16(x, device), t_qw(trip, 4, device), residual=t_bf16(r, device), **kw)
        want = affine.bf16_round(affine.bf16_round(want) + r)
    assert native.last_variant().startswith("qmv_w16" if w16 else "qmv_"), native.last_variant()
    assert w16 or not native.last_variant().startswith("qmv_w16"), native.last_variant()
    assert_close(n_f32(got), want, what=f"few rows {M}x{N}x{K}")


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K", [(8, 1000, 4096), (3, 96, 14336), (16, 2080, 2048), (5, 14336, 512)])
def test_qmv_swiglu_rows_equal_separate_launches(device, bits, M, N, K):
    """The one-launch (gate, up, SwiGLU) of 2..16 rows rounds each projection to bf16
    before the SwiGLU, so it equals the two GEMVs followed by the elementwise kernel bit
    for bit; with and without the fused RMSNorm, with K split over workgroups (short N)
    and not."""
    g = t_qw(rand_quantized(N, K, bits, seed=N + 1), bits, device)
    u = t_qw(rand_quantized(N, K, bits, seed=N + 2), bits, device)
    x = t_bf16(rand_bf16((M, K), seed=M + K, scale=2.0), device)
    w = t_bf16(affine.bf16_round(rand_bf16((K,), seed=6) * 0.1 + 1.0), device)
    for nw in (None, w):
        fused = ops.qmv_swiglu(x, g, u, norm_weight=nw, eps=1e-5)
        sep = ops.swiglu(ops.quantized_matmul(x, g, norm_weight=nw, eps=1e-5),
                         ops.quantized_matmul(x, u, norm_weight=nw, eps=1e-5))
        if (nw is None and M > 8 and bits == 8) or N * K * bits // 8 <= (1 << 20):
            # these single projections take the split-K GEMM, or (a matrix of up to 1 MiB)
            # one single-row launch set per row: another summation order
            assert_close(n_f32(fused), n_f32(sep), what="fused pair vs separate projections")
        else:
            assert torch.equal(fused.view(torch.int16), sep.view(torch.int16))
    # the shared workspace is left clean for a launch of another shape
    y = ops.quantized_matmul(x[:2], g)
    assert torch.equal(y.view(torch.int16), ops.quantized_matmul(x[:2], g).view(torch.int16))


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M", [2, 4, 8, 16])
@pytest.mark.parametrize("N,K", [(128, 2048), (60, 4096), (256, 768)])
def test_small_matrix_rows_equal_single_row_launches(device, bits, M, N, K):
    """A matrix of up to 1 MiB (a MoE router) under 2..16 rows runs the single-row kernel once
    per row in one launch: every row equals its own single-row launch bit for bit, with and
    without the fused RMSNorm, and the oracle within tolerance."""
    trip = rand_quantized(N, K, bits, seed=N + K)
    x = rand_bf16((M, K), seed=M + 7, scale=2.0)
    qw, xt = t_qw(trip, bits, device), t_bf16(x, device)
    w = t_bf16(affine.bf16_round(rand_bf16((K,), seed=6) * 0.1 + 1.0), device)
    for nw in (None, w):
        got = ops.quantized_matmul(xt, qw, norm_weight=nw, eps=1e-5)
        for r in range(M):
            one = ops.quantized_matmul(xt[r:r + 1], qw, norm_weight=nw, eps=1e-5)
            assert torch.equal(got[r:r + 1].view(torch.int16), one.view(torch.int16)), (r, nw is None)
    assert_close(n_f32(ops.quantized_matmul(xt, qw)), affine.qmm(x, *trip, 64, bits), what="rows of a small matrix")


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K", [(300, 256, 512), (129, 100, 192), (513, 192, 1024), (40, 64, 256), (2046, 1000, 320),
                                   (300, 4100, 768), (700, 8200, 768), (260, 4104, 1280)])
def test_qmm_swiglu_pair(device, bits, M, N, K):
    """Gate and up projections with the SwiGLU in the GEMM's epilogue: the bits of the two
    GEMMs followed by the elementwise kernel (same products, same rounding points), and the
    oracle within tolerance.  Ragged M and N, N not a multiple of 8, K with and without the
    four-step scale blocks; the last three shapes are launches of more than 128 tall tiles,
    which take the 128 x 128 tile with the four waves side by side."""
    g = rand_quantized(N, K, bits, seed=N + 11)
    u = rand_quantized(N, K, bits, seed=N + 12)
    x = rand_bf16((M, K), seed=M + K)
    gq, uq, xt = t_qw(g, bits, device), t_qw(u, bits, device), t_bf16(x, device)
    got = ops.qmm_swiglu(xt, gq, uq)
    sep = ops.swiglu(ops.qmm(xt, gq), ops.qmm(xt, uq))
    assert torch.equal(got.view(torch.int16), sep.view(torch.int16))
    # two roundings in a row (projection, then SwiGLU): a flipped bf16 rounding of a
    # projection near zero can leave a handful of the elements outside the elementwise
    # bound, so a fraction of 1e-5 is allowed
    want = O.swiglu(affine.qmm(x, *g, 64, bits), affine.qmm(x, *u, 64, bits))
    assert_close_stat(n_f32(got), want, max_outlier_frac=1e-5, what="qmm_swiglu")


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K", [(126, 8192, 2048), (40, 256, 1024), (100, 100, 768), (128, 4100, 4096), (17, 64, 512)])
def test_qmm_swiglu_pair_split_k(device, bits, M, N, K):
    """The pair GEMM of a short input with K split over workgroups (partials of both
    projections, then one reduce + SwiGLU launch): against the oracle, and against the unsplit
    launch (same rounding points, the float32 sums in another order), twice in a row on the
    shared workspace."""
    g = rand_quantized(N, K, bits, seed=N + 21)
    u = rand_quantized(N, K, bits, seed=N + 22)
    x = rand_bf16((M, K), seed=M + K + 1)
    gq, uq, xt = t_qw(g, bits, device), t_qw(u, bits, device), t_bf16(x, device)
    assert native.load().exo_qmm_swiglu_workspace(M, N) > 0
    one = ops.qmm_swiglu(xt, gq, uq, split_k=False)
    want = O.swiglu(affine.qmm(x, *g, 64, bits), affine.qmm(x, *u, 64, bits))
    for _ in range(2):
        got = ops.qmm_swiglu(xt, gq, uq)
        assert_close_stat(n_f32(got), want, max_outlier_frac=1e-5, what="qmm_swiglu split-K")
        assert_close_stat(n_f32(got), n_f32(one), max_outlier_frac=1e-4, what="split-K vs one launch")
        ops.qmm(xt, gq)  # another user of the workspace pool in between


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K", [(128, 256, 512), (33, 130, 192), (257, 128, 1024), (17, 64, 64)])
def test_qmm_mfma(device, bits, M, N, K):
    trip = rand_quantized(N, K, bits, seed=M + N)
    x = rand_bf16((M, K), seed=M * 3 + 1)
    got = n_f32(ops.qmm(t_bf16(x, device), t_qw(trip, bits, device)))
    want = affine.qmm(x, *trip, 64, bits)
    assert_close(got, want, what=f"qmm {M}x{N}x{K} b{bits}")


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K", [(100, 256, 4096), (33, 130, 14336), (128, 1000, 2048), (17, 64, 1024),
                                   (12, 256, 8192), (9, 96, 1024), (1023, 128, 2048), (300, 200, 4096),
                                   (32, 520, 512), (64, 600, 1024), (65, 300, 768), (20, 257, 256),
                                   (300, 10880, 1024), (1023, 2048, 1024), (300, 4100, 4096), (100, 14336, 4096),
                                   (600, 2052, 4096)])
def test_qmm_split_k(device, bits, M, N, K):
    """Few output tiles (a short input, or a narrow matrix under a long one): K is split
    over workgroups and the float32 partial tiles are added by a second launch.  Against
    the oracle, against the
    unsplit kernel (same products, another summation order: a few bf16 ulps at most),
    with the residual, and three times in a row with identical bits.  The last three
    shapes have K ranges of 1024 and take the wide tile with eight waves (two teams on the
    halves of a range)."""
    trip = rand_quantized(N, K, bits, seed=M + N)
    x = rand_bf16((M, K), seed=M * 3 + 1)
    r = rand_bf16((M, N), seed=M + 5)
    qw, xt, rt = t_qw(trip, bits, device), t_bf16(x, device), t_bf16(r, device)
    want = affine.qmm(x, *trip, 64, bits)
    first = None
    for _ in range(3):
        got = ops.quantized_matmul(xt, qw)
        assert_close(n_f32(got), want, what=f"qmm split-K {M}x{N}x{K} b{bits}")
        first = got.clone() if first is None else first
        assert torch.equal(got.view(torch.int16), first.view(torch.int16))
    unsplit = ops.qmm(xt, qw)
    assert_close(n_f32(got), n_f32(unsplit), rtol=1e-2, what="split vs unsplit")
    got_r = n_f32(ops.quantized_matmul(xt, qw, residual=rt))
    assert_close(got_r, affine.bf16_round(affine.bf16_round(want) + r), what="qmm split-K + residual")


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K", [(1100, 4100, 1024), (1300, 2052, 1536), (700, 8192, 1024)])
def test_qmm_eight_wave_tiles(device, bits, M, N, K):
    """Launches of more than 128 tall tiles but at most one tile per CU run eight waves per
    tile, two teams on the two halves of K merged through LDS: the wide 128 x 256 tile with
    the ring of four (4-bit) or the 256 x 128 tile (8-bit).  Ragged M and N, with the residual."""
    trip = rand_quantized(N, K, bits, seed=M + N)
    x = rand_bf16((M, K), seed=M * 3 + 1)
    r = rand_bf16((M, N), seed=M + 5)
    qw, xt, rt = t_qw(trip, bits, device), t_bf16(x, device), t_bf16(r, device)
    want = affine.qmm(x, *trip, 64, bits)
    assert_close(n_f32(ops.qmm(xt, qw)), want, what=f"qmm {M}x{N}x{K} b{bits}")
    got_r = n_f32(ops.quantized_matmul(xt, qw, residual=rt))
    assert_close(got_r, affine.bf16_round(affine.bf16_round(want) + r), what="qmm + residual")


def test_qmm_residual_and_dispatch(device):
    M, N, K, bits = 40, 192, 256, 4
    trip = rand_quantized(N, K, bits, seed=5)
    x = rand_bf16((M, K), seed=6)
    r = rand_bf16((M, N), seed=7)
    got = n_f32(ops.quantized_matmul(t_bf16(x, device), t_qw(trip, bits, device), residual=t_bf16(r, device)))
    want = affine.bf16_round(affine.qmm(x, *trip, 64, bits) + r)
    assert_close(got, want, what="qmm+residual")


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("x_rows", ["one", "topk"])
def test_gather_qmv(device, bits, x_rows):
    E, N, K, T, topk = 6, 96, 768, 3, 4
    trip = rand_quantized(N, K, bits, seed=40, E=E)
    idx = rng(41).integers(0, E, size=(T, topk)).astype(np.int32)
    R = 1 if x_rows == "one" else topk
    x = rand_bf16((T, R, K), seed=42)
    got = n_f32(ops.gather_qmm(t_bf16(x, device), t_qw(trip, bits, device), torch.from_numpy(idx).to(device)))
    want = affine.gather_qmm(x, *trip, idx, 64, bits)
    assert_close(got, want, what="gather_qmv")


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("x_rows", ["one", "topk"])
@pytest.mark.parametrize("E,N,K,T,topk", [(6, 96, 768, 40, 4), (128, 200, 128, 300, 8), (3, 64, 64, 1, 2)])
def test_grouped_qmm(device, bits, x_rows, E, N, K, T, topk):
    """Prefill-sized gather_qmm: pairs sorted by expert, one matrix-core tile row block per
    expert run (experts with no rows, with a partial tile and with several tiles), against
    the oracle's per-pair loop."""
    trip = rand_quantized(N, K, bits, seed=40 + E, E=E)
    idx = rng(41 + T).integers(0, E, size=(T, topk)).astype(np.int32)
    if E == 128:
        idx[: T // 2, 0] = 5  # one expert with more than a tile of rows
    R = 1 if x_rows == "one" else topk
    x = rand_bf16((T, R, K), seed=42)
    it = torch.from_numpy(idx).to(device)
    ws = ops.moe_group(it, E)
    P = T * topk
    sorted_pairs = ws[:P].cpu().numpy()
    assert sorted(sorted_pairs.tolist()) == list(range(P))          # a permutation of the pairs
    experts_in_order = idx.reshape(-1)[sorted_pairs]
    assert np.all(np.diff(experts_in_order) >= 0)                    # grouped by expert
    tiles = ws[P:].cpu().numpy().reshape(-1, 3)
    used = tiles[tiles[:, 0] >= 0]
    assert used[:, 2].sum() == P and used[:, 2].max() <= 128
    got = n_f32(ops.grouped_qmm(t_bf16(x, device), t_qw(trip, bits, device), ws, topk))
    want = affine.gather_qmm(x, *trip, idx, 64, bits)
    assert_close(got, want, what="grouped_qmm")


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("E,N,K,T,topk", [(6, 96, 768, 40, 4), (128, 200, 256, 300, 8), (3, 60, 64, 1, 2)])
def test_grouped_qmm_swiglu(device, bits, E, N, K, T, topk):
    """SwitchGLU's gate and up projections with the SwiGLU in the grouped GEMM's epilogue:
    the bits of the two grouped GEMMs followed by the elementwise kernel (ragged tiles,
    N not a multiple of 64 or 8, K with and without the four-step scale blocks)."""
    g = rand_quantized(N, K, bits, seed=60 + E, E=E)
    u = rand_quantized(N, K, bits, seed=61 + E, E=E)
    idx = rng(62 + T).integers(0, E, size=(T, topk)).astype(np.int32)
    if E == 128:
        idx[: T // 2, 0] = 5
    x = t_bf16(rand_bf16((T, 1, K), seed=63), device)
    gq, uq = t_qw(g, bits, device), t_qw(u, bits, device)
    ws = ops.moe_group(torch.from_numpy(idx).to(device), E)
    got = ops.grouped_qmm_swiglu(x, gq, uq, ws, topk)
    sep = ops.swiglu(ops.grouped_qmm(x, gq, ws, topk), ops.grouped_qmm(x, uq, ws, topk))
    assert torch.equal(got.view(torch.int16), sep.view(torch.int16))


@pytest.mark.parametrize("bits", [4, 8])
def test_gather_qmv_swiglu(device, bits):
    E, N, K, T, topk = 5, 64, 2048, 2, 3
    g = rand_quantized(N, K, bits, seed=50, E=E)
    u = rand_quantized(N, K, bits, seed=51, E=E)
    idx = rng(52).integers(0, E, size=(T, topk)).astype(np.int32)
    x = rand_bf16((T, K), seed=53)
    got = n_f32(ops.gather_qmv_swiglu(t_bf16(x, device), t_qw(g, bits, device), t_qw(u, bits, device), torch.from_numpy(idx).to(device)))
    want = O.swiglu(affine.gather_qmm(x[:, None], *g, idx, 64, bits), affine.gather_qmm(x[:, None], *u, idx, 64, bits))
    assert_close(got, want, what="gather_qmv_swiglu")


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("E,N,K,T,topk,renorm,norm", [(128, 768, 2048, 1, 8, True, True), (128, 768, 2048, 4, 8, True, True),
                                                      (60, 64, 2048, 3, 4, False, False), (256, 96, 512, 2, 16, True, True),
                                                      (7, 200, 768, 5, 3, True, False)])
def test_route_gather_qmv_swiglu_equals_topk_then_gather(device, bits, E, N, K, T, topk, renorm, norm):
    """The expert gate/up launch that routes by itself: the indices and scores it writes are
    those of exo_router_topk bit for bit, its output that of the gather launch given them
    (row-streaming and generic kernel, with and without the fused norm); indices also against
    the oracle."""
    g = rand_quantized(N, K, bits, seed=70 + E, E=E)
    u = rand_quantized(N, K, bits, seed=71 + E, E=E)
    logits = rand_bf16((T, E), seed=72 + E, scale=2.0)
    x = t_bf16(rand_bf16((T, K), seed=73), device)
    nw = t_bf16(affine.bf16_round(rand_bf16((K,), seed=74) + 1.0), device) if norm else None
    gq, uq, lt = t_qw(g, bits, device), t_qw(u, bits, device), t_bf16(logits, device)
    idx0, sc0 = ops.router_topk(lt, topk, renorm)
    want = ops.gather_qmv_swiglu(x, gq, uq, idx0, norm_weight=nw, eps=1e-5)
    for _ in range(2):
        idx, sc, got = ops.route_gather_qmv_swiglu(x, lt, topk, renorm, gq, uq, norm_weight=nw, eps=1e-5)
        assert torch.equal(idx, idx0)
        assert torch.equal(sc.view(torch.int16), sc0.view(torch.int16))
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    np.testing.assert_array_equal(idx0.cpu().numpy(), O.router_topk(logits, topk, renorm)[0])


def test_bad_arguments_raise(device):
    trip = rand_quantized(64, 128, 4, seed=1)
    qw = t_qw(trip, 4, device)
    with pytest.raises(ValueError):
        ops.quantized_matmul(t_bf16(rand_bf16((1, 64), 1), device), qw)
    lib = native.load()
    assert lib.exo_qmv(None, None, None, None, None, None, 1, 64, 128, 5, 64, None) == -1
    assert b"bits" in lib.exo_last_error()
    assert lib.exo_qmv(None, None, None, None, None, None, 1, 64, 128, 4, 32, None) == -1
    assert lib.exo_qmv(None, None, None, None, None, None, 17, 64, 128, 4, 64, None) == -1


@pytest.mark.parametrize("H", [2048, 4096, 64, 8192])
@pytest.mark.parametrize("with_res", [False, True])
def test_add_rmsnorm(device, H, with_res):
    rows = 5
    x = rand_bf16((rows, H), seed=H)
    r = rand_bf16((rows, H), seed=H + 1) if with_res else None
    w = rand_bf16((H,), seed=H + 2) + 1.0
    w = affine.bf16_round(w)
    h, n = ops.add_rms_norm(t_bf16(x, device), t_bf16(r, device) if with_res else None, t_bf16(w, device), 1e-5)
    hh = affine.bf16_round(x + r) if with_res else x
    np.testing.assert_array_equal(n_f32(h), hh)
    assert_close(n_f32(n), O.rms_norm(hh, w, 1e-5), rtol=1e-2, what="rmsnorm")


@pytest.mark.parametrize("D,Hq,Hkv", [(64, 8, 2), (128, 4, 4), (128, 16, 2)])
@pytest.mark.parametrize("qk_norm", [False, True])
def test_rope_kv_append(device, D, Hq, Hkv, qk_norm):
    B, T, S_max = 2, 3, 40
    pos = np.array([5, 17], np.int32)
    qkv = rand_bf16((B * T, (Hq + 2 * Hkv) * D), seed=D + Hq)
    scaling = {"rope_type": "llama3", "factor": 8.0, "low_freq_factor": 1.0, "high_freq_factor": 4.0, "original_max_position_embeddings": 8192}
    inv = O.rope_inv_freq(D, 5e5, scaling)
    qn = affine.bf16_round(rand_bf16((D,), 3) + 1.0) if qk_norm else None
    kn = affine.bf16_round(rand_bf16((D,), 4) + 1.0) if qk_norm else None
    kc = torch.zeros(B, Hkv, S_max, D, dtype=torch.bfloat16, device=device)
    vc = torch.zeros_like(kc)
    q_out = torch.empty(B * T, Hq * D, dtype=torch.bfloat16, device=device)
    ops.rope_kv_append(
        t_bf16(qkv, device), q_out, kc, vc, torch.from_numpy(pos).to(device),
        torch.from_numpy(inv).to(device), B, T, Hq, Hkv, D,
        t_bf16(qn, device) if qk_norm else None, t_bf16(kn, device) if qk_norm else None, 1e-6,
    )
    x = qkv.reshape(B, T, Hq + 2 * Hkv, D)
    q, k, v = x[:, :, :Hq], x[:, :, Hq:Hq + Hkv], x[:, :, Hq + Hkv:]
    if qk_norm:
        q = O.rms_norm(q, qn, 1e-6)
        k = O.rms_norm(k, kn, 1e-6)
    for b in range(B):
        qr = O.rope(q[b:b + 1].transpose(0, 2, 1, 3), inv, int(pos[b]))  # [1,H,T,D]
        kr = O.rope(k[b:b + 1].transpose(0, 2, 1, 3), inv, int(pos[b]))
        got_q = n_f32(q_out).reshape(B, T, Hq, D)[b].transpose(1, 0, 2)
        assert_close(got_q, qr[0], rtol=1e-2, what="rope q")
        got_k = n_f32(kc)[b, :, pos[b]:pos[b] + T]
        assert_close(got_k, kr[0], rtol=1e-2, what="rope k")
        np.testing.assert_array_equal(n_f32(vc)[b, :, pos[b]:pos[b] + T], v[b].transpose(1, 0, 2))
    # nothing outside the appended window was written
    assert float(n_f32(kc)[0, :, :5].sum()) == 0.0 and float(n_f32(kc)[0, :, 8:].sum()) == 0.0
    # with the angle table (long enough; too short for the second sequence): the same bits
    inv_t = torch.from_numpy(inv).to(device)
    for rows in (S_max, 12):
        kc2, vc2, q2 = torch.zeros_like(kc), torch.zeros_like(vc), torch.empty_like(q_out)
        ops.rope_kv_append(
            t_bf16(qkv, device), q2, kc2, vc2, torch.from_numpy(pos).to(device), inv_t, B, T, Hq, Hkv, D,
            t_bf16(qn, device) if qk_norm else None, t_bf16(kn, device) if qk_norm else None, 1e-6,
            rope_tab=ops.rope_table(inv_t, rows, D),
        )
        for a, b_ in ((q2, q_out), (kc2, kc), (vc2, vc)):
            assert torch.equal(a.view(torch.int16), b_.view(torch.int16))


@pytest.mark.parametrize("rows,H", [(1, 8), (3, 2048), (2, 2056), (5, 4096), (2, 4104), (3, 6144), (2, 6152), (61, 8192),
                                    (800, 2056), (1023, 4096), (2100, 2064), (800, 4104), (1600, 6144), (1800, 8192), (2442, 2048)])
@pytest.mark.parametrize("residual", [False, True])
def test_add_rms_norm_chunks(device, rows, H, residual):
    """One to four pieces of a row per thread, full and not, requested together and one after another; the sum in place of the residual."""
    g = torch.Generator(device=device).manual_seed(H)
    x, r = (torch.randn(rows, H, device=device, generator=g).bfloat16() for _ in range(2))
    w = (1 + 0.1 * torch.randn(H, device=device, generator=g)).bfloat16()
    h = (x.float() + r.float()).bfloat16() if residual else x
    sum_, got = ops.add_rms_norm(x, r if residual else None, w, 1e-5, r if residual else None)
    assert torch.equal(sum_, h)
    want = h.double() * (h.double().pow(2).mean(1, keepdim=True) + 1e-5).rsqrt() * w.double()
    assert bool(((got.double() - want).abs() <= (2.0**-8 + (H / 4 + 10) * 2.0**-24) * want.abs()).all())


@pytest.mark.parametrize("D,Hq,Hkv", [(64, 5, 1), (64, 6, 1), (64, 7, 1), (64, 14, 1), (64, 15, 1), (64, 96, 1), (128, 46, 1), (128, 64, 8), (128, 1, 1), (128, 2, 1), (128, 3, 1), (128, 6, 1), (128, 7, 1)])
@pytest.mark.parametrize("qk_norm", [False, True])
def test_rope_kv_append_pieces(device, D, Hq, Hkv, qk_norm):
    """Operands at 16 bytes against ones that are not, which go element by element: the same bits, with head norms but for the order of
    a sum of squares (an element's rounding to bf16, once ahead of the rotation and once behind it); positions past the table and past the cache."""
    B, T, S_max, rows = 2, 37, 60, 45
    g = torch.Generator(device=device).manual_seed(D + Hq)
    n = B * T * (Hq + 2 * Hkv) * D
    flat = torch.randn(n + 8, device=device, generator=g).bfloat16()
    qn, kn = ((1 + 0.1 * torch.randn(D, device=device, generator=g)).bfloat16() for _ in range(2))
    inv = torch.from_numpy(O.rope_inv_freq(D, 5e5, None)).to(device)
    pos = torch.tensor([0, 30], dtype=torch.int32, device=device)
    out = []
    for at in (0, 4):
        qkv = (flat[8:].clone() if at == 0 else torch.cat((flat[:4], flat[8:]))[at:]).view(B * T, -1)
        assert (qkv.data_ptr() % 16 == 0) == (at == 0)
        kc, vc = (torch.full((B, Hkv, S_max, D), 7.0, device=device).bfloat16() for _ in range(2))
        q = torch.empty(B * T, Hq * D, device=device).bfloat16()
        ops.rope_kv_append(qkv, q, kc, vc, pos, inv, B, T, Hq, Hkv, D, qn if qk_norm else None, kn if qk_norm else None, 1e-6,
                           rope_tab=ops.rope_table(inv, rows, D))
        out.append((q.float().view(B, T, Hq, D), kc.float(), vc.float()))
    for i, (a, b) in enumerate(zip(*out)):
        size = a.abs() + torch.cat((a[..., D // 2 :], a[..., : D // 2]), -1).abs()
        assert bool(((a - b).abs() <= (2.0**-6 * size if qk_norm and i < 2 else 0.0)).all())
    assert bool((out[0][1][0, :, T:] == 7).all()) and bool((out[0][2][1, :, :30] == 7).all())


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("at", [0, 4])
def test_rope_kv_append_rows_without_a_table(device, D, at):
    """A null table with a number of rows, operands at 16 bytes and not: the angles come from the frequencies for every position, as
    in the entry point that takes no table."""
    B, T, Hq, Hkv, S_max = 2, 5, 4, 2, 16
    g = torch.Generator(device=device).manual_seed(D)
    n = B * T * (Hq + 2 * Hkv) * D
    qkv = torch.randn(n + 8, device=device, generator=g).bfloat16()[at : at + n]
    inv = torch.from_numpy(O.rope_inv_freq(D, 5e5, None)).to(device)
    pos = torch.tensor([0, 9], dtype=torch.int32, device=device)
    out = []
    for rows in (None, 8):
        kc, vc = (torch.zeros(B, Hkv, S_max, D, device=device).bfloat16() for _ in range(2))
        q = torch.empty(B * T, Hq * D, device=device).bfloat16()
        head = [t.data_ptr() for t in (qkv, q, kc, vc, pos, inv)]
        tail = [None, None, 0.0, B, T, Hq, Hkv, D, S_max, torch.cuda.current_stream().cuda_stream]
        lib = native.load()
        rc = lib.exo_rope_kv_append(*head, *tail) if rows is None else lib.exo_rope_kv_append_tab(*head, None, rows, *tail)
        assert rc == 0
        out.append((q, kc, vc))
    for a, b in zip(*out):
        assert torch.equal(a, b) and bool(a.any())


@pytest.mark.parametrize("D,Hq,Hkv", [(64, 32, 8), (128, 32, 8), (128, 32, 4), (128, 64, 4), (128, 4, 4)])
@pytest.mark.parametrize("lens", [[1, 2], [100, 37], [513, 1024]])
def test_sdpa_decode(device, D, Hq, Hkv, lens):
    B, S_max = len(lens), 1024
    q = rand_bf16((B, Hq * D), seed=D + Hq + lens[0])
    k = rand_bf16((B, Hkv, S_max, D), seed=11)
    v = rand_bf16((B, Hkv, S_max, D), seed=12)
    pos = np.array([n - 1 for n in lens], np.int32)
    out = torch.empty(B, Hq * D, dtype=torch.bfloat16, device=device)
    ws = ops.sdpa_decode_workspace(B, Hq, D, device)
    ops.sdpa_decode(t_bf16(q, device), t_bf16(k, device), t_bf16(v, device), torch.from_numpy(pos).to(device), out, ws, D ** -0.5, B, Hq, Hkv, D)
    for b in range(B):
        want = O.sdpa(q[b].reshape(1, Hq, 1, D), k[b:b + 1, :, :lens[b]], v[b:b + 1, :, :lens[b]], D ** -0.5, None)
        assert_close(n_f32(out)[b].reshape(Hq, D), want[0, :, 0], what=f"sdpa decode len {lens[b]}")


@pytest.mark.parametrize("D,Hq,Hkv", [(64, 8, 2), (128, 8, 2), (128, 4, 4), (128, 4, 2), (128, 16, 2), (64, 16, 1)])
@pytest.mark.parametrize("T,pos", [(19, (0, 30)), (5, (0, 3)), (100, (0, 77)), (64, (64, 1)), (161, (0, 200))])
def test_sdpa_prefill_causal(device, D, Hq, Hkv, T, pos):
    """Chunks shorter than 8 tokens run the per-token kernel, longer ones the matrix-core
    flash kernel: 1, 2, 4, 8 and 16 query heads per kv head, chunk lengths on and off the
    32-token tile, caches that start empty and part-filled, several key tiles."""
    B, S_max = 2, 384
    pos = np.array(pos, np.int32)
    q = rand_bf16((B * T, Hq * D), seed=D + T)
    k = rand_bf16((B, Hkv, S_max, D), seed=13)
    v = rand_bf16((B, Hkv, S_max, D), seed=14)
    out = torch.empty(B * T, Hq * D, dtype=torch.bfloat16, device=device)
    ops.sdpa_prefill(t_bf16(q, device), t_bf16(k, device), t_bf16(v, device), torch.from_numpy(pos).to(device), out, D ** -0.5, B, T, Hq, Hkv, D)
    for b in range(B):
        S = int(pos[b]) + T
        qq = q.reshape(B, T, Hq, D)[b:b + 1].transpose(0, 2, 1, 3)
        want = O.sdpa(qq, k[b:b + 1, :, :S], v[b:b + 1, :, :S], D ** -0.5, S - T)
        got = n_f32(out).reshape(B, T, Hq, D)[b].transpose(1, 0, 2)
        assert_close(got, want[0], what=f"sdpa prefill T={T} pos={pos[b]}")


def test_sdpa_prefill_cache_exactly_full(device):
    """The last key tile ends at the end of the cache allocation (no reads past it)."""
    B, T, Hq, Hkv, D, S_max = 1, 40, 8, 2, 128, 100
    pos = np.array([60], np.int32)
    q = rand_bf16((B * T, Hq * D), seed=3)
    k = rand_bf16((B, Hkv, S_max, D), seed=4)
    v = rand_bf16((B, Hkv, S_max, D), seed=5)
    out = torch.empty(B * T, Hq * D, dtype=torch.bfloat16, device=device)
    ops.sdpa_prefill(t_bf16(q, device), t_bf16(k, device), t_bf16(v, device), torch.from_numpy(pos).to(device), out, D ** -0.5, B, T, Hq, Hkv, D)
    qq = q.reshape(B, T, Hq, D).transpose(0, 2, 1, 3)
    want = O.sdpa(qq, k, v, D ** -0.5, S_max - T)
    assert_close(n_f32(out).reshape(T, Hq, D).transpose(1, 0, 2), want[0], what="sdpa prefill full cache")


def test_swiglu(device):
    g = rand_bf16((3, 1001), seed=1, scale=3.0)
    u = rand_bf16((3, 1001), seed=2)
    got = n_f32(ops.swiglu(t_bf16(g, device), t_bf16(u, device)))
    assert_close(got, O.swiglu(g, u), rtol=1e-2, what="swiglu")


@pytest.mark.parametrize("E,k,renorm", [(128, 8, True), (128, 8, False), (60, 4, True), (256, 16, True)])
def test_router_topk(device, E, k, renorm):
    rows = 9
    logits = rand_bf16((rows, E), seed=E + k, scale=2.0)
    idx, sc = ops.router_topk(t_bf16(logits, device), k, renorm)
    widx, wsc = O.router_topk(logits, k, renorm)
    np.testing.assert_array_equal(idx.cpu().numpy(), widx)
    assert_close(n_f32(sc), wsc, rtol=2.0**-7, what="router scores")


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("E,N,K,T,topk", [(6, 200, 768, 3, 8), (5, 96, 1536, 2, 4), (4, 64, 2048, 1, 2),
                                          (3, 72, 192, 2, 3), (9, 64, 768, 2, 9)])
def test_gather_qmv_combine(device, bits, E, N, K, T, topk):
    """Down projection of SwitchGLU + weighted sum over the experts + residual in one
    launch: against the oracle, and against the two separate launches it replaces
    (same rounding points; the dot products are summed in another order).  The last two
    shapes take the fallback through the scratch buffer (rows that share a wave by
    threes; more than 8 experts per token)."""
    trip = rand_quantized(N, K, bits, seed=E + N, E=E)
    idx = rng(43).integers(0, E, size=(T, topk)).astype(np.int32)
    x = rand_bf16((T, topk, K), seed=44)
    sc = affine.bf16_round(np.abs(rand_bf16((T, topk), seed=45)) / 8)
    r = rand_bf16((T, N), seed=46)
    qw, xt, it = t_qw(trip, bits, device), t_bf16(x, device), torch.from_numpy(idx).to(device)
    st, rt = t_bf16(sc, device), t_bf16(r, device)
    scratch = torch.empty(T, topk, N, dtype=torch.bfloat16, device=device)
    got = ops.gather_qmv_combine(xt, qw, it, st, residual=rt, scratch=scratch)
    eo = affine.gather_qmm(x, *trip, idx, 64, bits)
    acc = affine.bf16_round(affine.bf16_round(eo * sc[..., None]).sum(1, dtype=np.float32))
    assert_close(n_f32(got), affine.bf16_round(acc + r), what="gather_qmv_combine")
    sep = ops.moe_combine(ops.gather_qmm(xt, qw, it), st, rt)
    assert_close(n_f32(got), n_f32(sep), rtol=1e-2, what="fused vs separate")
    no_res = ops.gather_qmv_combine(xt, qw, it, st, scratch=scratch)
    assert_close(n_f32(no_res), acc, what="gather_qmv_combine without residual")


@pytest.mark.parametrize("bits,N,K,T,topk,tiles", [
    (4, 5, 768, 1, 8, 1), (4, 2053, 768, 3, 8, 2), (4, 4099, 1024, 5, 3, 4), (4, 8203, 1536, 6, 8, 8), (4, 523, 2048, 2, 6, 1),
    (8, 9, 512, 1, 1, 1), (8, 6149, 768, 1, 5, 2), (8, 4110, 1024, 6, 2, 8), (8, 4093, 1536, 3, 8, 4),
])
def test_gather_qmv_combine_planes(device, bits, N, K, T, topk, tiles):
    """The down projection on the integer matrix cores: last tiles of a few rows, one to eight tiles per wave, every length of a
    half row; against the two launches that it stands for, and an element that is not a number."""
    g = torch.Generator(device=device).manual_seed(N + K)
    E = max(topk, 4)
    w = torch.randint(-2**31, 2**31 - 1, (E, N, K * bits // 32), dtype=torch.int32, device=device, generator=g)
    s, b = (torch.randn(E, N, K // 64, device=device, generator=g).bfloat16() * f for f in (0.02, 0.1))
    qw = ops.QuantizedWeight(w, s, b, bits)
    x = (torch.randn(T, topk, K, device=device, generator=g) * torch.exp(2 * torch.randn(T, topk, K, device=device, generator=g))).bfloat16()
    idx = torch.stack([torch.randperm(E, generator=torch.Generator().manual_seed(t))[:topk] for t in range(T)]).int().to(device)
    sc = torch.rand(T, topk, device=device, generator=g).bfloat16()
    r = torch.randn(T, N, device=device, generator=g).bfloat16()
    scratch = torch.empty(T, topk, N, dtype=torch.bfloat16, device=device)
    got = ops.gather_qmv_combine(x, qw, idx, sc, residual=r, scratch=scratch)
    assert native.last_variant().startswith(f"moe_down_planes<{bits},") and f" tiles={tiles} " in native.last_variant(), native.last_variant()
    want = ops.moe_combine(ops.gather_qmm(x, qw, idx), sc, r)
    assert_close(n_f32(got), n_f32(want), rtol=1e-2, what="planes")
    x[0, topk - 1, K - 1] = float("nan")
    bad = ops.gather_qmv_combine(x, qw, idx, sc, residual=r, scratch=scratch)
    assert bad[0].isnan().all() and torch.equal(bad[1:], got[1:])


@pytest.mark.parametrize("T,topk,H", [(3, 8, 2048), (5, 6, 4096), (2, 3, 100), (4, 9, 264)])
def test_moe_combine(device, T, topk, H):
    """Rows of 8-element multiples take the 16-byte kernel (slots in groups of four, the
    last group partial), the others the scalar one."""
    y = rand_bf16((T, topk, H), seed=1)
    s = affine.bf16_round(np.abs(rand_bf16((T, topk), seed=2)) / 8)
    r = rand_bf16((T, H), seed=3)
    got = n_f32(ops.moe_combine(t_bf16(y, device), t_bf16(s, device), t_bf16(r, device)))
    acc = affine.bf16_round(affine.bf16_round(y * s[..., None]).sum(1, dtype=np.float32))
    assert_close(got, affine.bf16_round(acc + r), rtol=1e-2, what="moe_combine")


@pytest.mark.parametrize("V", [128256, 1000, 64])
def test_argmax_logsumexp(device, V):
    rows = 3
    logits = rand_bf16((rows, V), seed=V, scale=2.0)
    logits[1, 7] = logits[1].max()  # a tie: lowest index must win
    tok = torch.empty(rows, dtype=torch.int32, device=device)
    lse = torch.empty(rows, dtype=torch.float32, device=device)
    lp = torch.empty(rows, dtype=torch.float32, device=device)
    pos = torch.tensor([4, 5, 6], dtype=torch.int32, device=device)
    ops.argmax_logsumexp(t_bf16(logits, device), tok, lse, lp, ops.argmax_workspace(rows, device), pos)
    np.testing.assert_array_equal(tok.cpu().numpy(), np.argmax(logits, -1))
    want_lse = O.logsumexp(logits)[:, 0]
    np.testing.assert_allclose(lse.cpu().numpy(), want_lse, rtol=1e-5)
    np.testing.assert_allclose(lp.cpu().numpy(), logits.max(-1) - want_lse, rtol=1e-4, atol=1e-5)
    assert pos.cpu().tolist() == [5, 6, 7]


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("N,K,M", [(256, 4096, 1), (128, 14336, 2), (96, 768, 1), (64, 2048, 4), (72, 192, 3),
                                   (200, 4096, 2), (64, 8192, 2)])
def test_norm_qmv_fused(device, bits, N, K, M):
    trip = rand_quantized(N, K, bits, seed=N + K)
    x = rand_bf16((M, K), seed=K + M, scale=3.0)
    w = affine.bf16_round(rand_bf16((K,), seed=5) * 0.1 + 1.0)
    got = n_f32(ops.quantized_matmul(t_bf16(x, device), t_qw(trip, bits, device), norm_weight=t_bf16(w, device), eps=1e-5))
    want = affine.qmm(O.rms_norm(x, w, 1e-5), *trip, 64, bits)
    assert_close(got, want, what="norm+qmv")
    g = rand_quantized(N, K, bits, seed=N + K + 1)
    got = n_f32(ops.qmv_swiglu(t_bf16(x, device), t_qw(trip, bits, device), t_qw(g, bits, device), norm_weight=t_bf16(w, device), eps=1e-5))
    xn = O.rms_norm(x, w, 1e-5)
    assert_close(got, O.swiglu(affine.qmm(xn, *trip, 64, bits), affine.qmm(xn, *g, 64, bits)), what="norm+qmv_swiglu")


@pytest.mark.parametrize("D,Hq,Hkv", [(64, 32, 8), (128, 32, 8), (128, 64, 4), (128, 4, 4), (128, 32, 4),
                                      (128, 16, 4)])
@pytest.mark.parametrize("qk_norm", [False, True])
@pytest.mark.parametrize("lens", [[1, 2], [100, 37], [513, 1000], [129, 33, 1024, 257]])
@pytest.mark.parametrize("table", [False, True])
def test_attn_decode_fused(device, D, Hq, Hkv, qk_norm, lens, table):
    """rope + head norm + cache append + attention in one launch == the three oracle ops."""
    B, S_max = len(lens), 1024
    pos = np.array([n - 1 for n in lens], np.int32)
    qkv = rand_bf16((B, (Hq + 2 * Hkv) * D), seed=D + Hq + lens[0])
    k = rand_bf16((B, Hkv, S_max, D), seed=11)
    v = rand_bf16((B, Hkv, S_max, D), seed=12)
    inv = O.rope_inv_freq(D, 5e5, {"rope_type": "llama3", "factor": 8.0, "low_freq_factor": 1.0,
                                   "high_freq_factor": 4.0, "original_max_position_embeddings": 8192})
    qn = affine.bf16_round(rand_bf16((D,), 3) * 0.1 + 1.0) if qk_norm else None
    kn = affine.bf16_round(rand_bf16((D,), 4) * 0.1 + 1.0) if qk_norm else None
    kc, vc = t_bf16(k, device), t_bf16(v, device)
    out = torch.empty(B, Hq * D, dtype=torch.bfloat16, device=device)
    ws = ops.sdpa_decode_workspace(B, Hq, D, device)
    inv_t = torch.from_numpy(inv).to(device)
    tab = ops.rope_table(inv_t, S_max, D) if table else None
    for _ in range(2):  # twice: the arrival counters must be back at zero
        ops.attn_decode(t_bf16(qkv, device), kc, vc, torch.from_numpy(pos).to(device),
                        inv_t, out, ws, D ** -0.5, B, Hq, Hkv, D,
                        t_bf16(qn, device) if qk_norm else None, t_bf16(kn, device) if qk_norm else None, 1e-6,
                        rope_tab=tab)
    x = qkv.reshape(B, 1, Hq + 2 * Hkv, D)
    q, kk, vv = x[:, :, :Hq], x[:, :, Hq:Hq + Hkv], x[:, :, Hq + Hkv:]
    if qk_norm:
        q, kk = O.rms_norm(q, qn, 1e-6), O.rms_norm(kk, kn, 1e-6)
    for b in range(B):
        p = int(pos[b])
        qr = O.rope(q[b:b + 1].transpose(0, 2, 1, 3), inv, p)
        kr = O.rope(kk[b:b + 1].transpose(0, 2, 1, 3), inv, p)
        kfull = np.concatenate([k[b:b + 1, :, :p], kr], axis=2)
        vfull = np.concatenate([v[b:b + 1, :, :p], vv[b:b + 1].transpose(0, 2, 1, 3)], axis=2)
        want = O.sdpa(qr, kfull, vfull, D ** -0.5, None)
        assert_close(n_f32(out)[b].reshape(Hq, D), want[0, :, 0], what=f"attn_decode len {lens[b]}")
        assert_close(n_f32(kc)[b, :, p], kr[0, :, 0], rtol=1e-2, what="appended k")
        np.testing.assert_array_equal(n_f32(vc)[b, :, p], vv[b, 0])
        np.testing.assert_array_equal(n_f32(kc)[b, :, p + 1:], k[b, :, p + 1:])  # nothing else touched
        np.testing.assert_array_equal(n_f32(kc)[b, :, :p], k[b, :, :p])


@pytest.mark.parametrize("Hq,Hkv", [(32, 8), (32, 4), (64, 4)])
@pytest.mark.parametrize("lens", [[1, 32, 33, 34], [192, 193, 194, 257], [319, 320, 321, 322], [481, 482, 641, 1024], [225, 226, 256, 258]])
def test_attn_decode_matrix_core_edges(device, Hq, Hkv, lens):
    """The matrix-core decode kernel where a tile, a round of its waves, one workgroup's share or a split ends."""
    test_attn_decode_fused(device, 128, Hq, Hkv, False, lens, True)
    assert native.last_variant().startswith(f"sdpa_decode_mfma<{Hq // Hkv}>"), native.last_variant()


# ------------------------------------------------------------------ KV wire layout


@pytest.mark.parametrize("Hkv,S_max,D,start,n", [(8, 64, 128, 0, 64), (4, 300, 64, 7, 201),
                                                 (2, 16, 8, 15, 1), (3, 40, 128, 5, 0)])
def test_kv_export_import_nhd(device, Hkv, S_max, D, start, n):
    """Byte-exact against the transpose the reference ships
    (engines/mlx/disaggregated/adapter.py:74-83): wire[t,h,:] = cache[h,start+t,:]."""
    g = torch.Generator(device="cpu").manual_seed(5)
    row = torch.randn(Hkv, S_max, D, generator=g).bfloat16().to(device)
    wire = ops.kv_export_nhd(row, start, n)
    want = row[:, start:start + n].permute(1, 0, 2).contiguous()
    assert wire.shape == (n, Hkv, D) and torch.equal(wire.view(torch.int16), want.view(torch.int16))
    dst = torch.full_like(row, 7.0)
    ops.kv_import_nhd(wire, dst, start)
    ref = torch.full_like(row, 7.0)
    ref[:, start:start + n] = row[:, start:start + n]
    assert torch.equal(dst.view(torch.int16), ref.view(torch.int16))


def test_kv_wire_argument_errors(device):
    row = torch.zeros(2, 16, 8, dtype=torch.bfloat16, device=device)
    with pytest.raises(ValueError):
        ops.kv_export_nhd(row, 10, 7)            # beyond S_max
    with pytest.raises(ValueError):
        ops.kv_export_nhd(row, -1, 2)
    with pytest.raises(ValueError):
        ops.kv_import_nhd(torch.zeros(3, 2, 4, dtype=torch.bfloat16, device=device), row, 0)
    with pytest.raises(ValueError):
        ops.kv_export_nhd(torch.zeros(2, 16, 12, dtype=torch.bfloat16, device=device), 0, 1)


def test_qmv_workspace_shared_by_launches_of_different_shapes(device):
    """The split-K workspace is shared by all 2..16-row GEMVs of a device: a launch with a
    short N must not leave anything where a later launch with more row blocks keeps its
    arrival counters (the partial sums sit behind a counter area of fixed size)."""
    for bits, M, N, K in [(4, 3, 128, 4096), (4, 16, 4096, 14336), (8, 5, 64, 2048), (8, 8, 4096, 14336),
                          (4, 16, 4096, 14336)]:
        trip = rand_quantized(64, K, bits, seed=N + K + bits)
        reps = N // 64
        trip = tuple(np.concatenate([t] * reps) for t in trip)  # N rows from 64 distinct ones
        x = rand_bf16((M, K), seed=M + K)
        got = n_f32(ops.quantized_matmul(t_bf16(x, device), t_qw(trip, bits, device)))
        want = np.tile(affine.qmm(x, *(t[:64] for t in trip), 64, bits), (1, reps))
        assert_close(got, want, what=f"qmv {M}x{N}x{K} b{bits}")


@pytest.mark.parametrize("n", [0, 1, 64, 65, 960, 961, 3840, 3841])
def test_put_ints(device, n):
    """Whole numbers from the host, in the launches' arguments or as a copy: exactly those, behind what the stream holds,
    whatever becomes of the host's memory, and nothing past them."""
    host = np.random.default_rng(n).integers(-2**31, 2**31, n).astype(np.int32)
    want = host.copy()
    buf = torch.full((n + 8,), 7, dtype=torch.int32, device=device)
    for _ in range(3):
        buf.fill_(9)
        ops.put_ints(buf[4 : 4 + n], host)
        host[:] = 0
        got = buf.cpu().numpy()
        assert (got[:4] == 9).all() and (got[4 + n :] == 9).all()
        np.testing.assert_array_equal(got[4 : 4 + n], want)
        host[:] = want
    with pytest.raises(ValueError):
        ops.put_ints(buf, list(range(n)))
