"""Products of few rows with few columns, whose parts of K lie side by side in one launch, against float64."""

from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
if not torch.cuda.is_available():
    pytest.skip("needs a GPU", allow_module_level=True)

from exo_amd import dense_ops as D, native  # noqa: E402


def check(got, x, w, bias=0.0):
    """A sum of K products in float32, in any order: at most K roundings of 2^-24 of the sum of their sizes."""
    x, w = x.double(), w.double()
    want, size = x @ w.T + bias, x.abs() @ w.abs().T
    bound = (x.shape[1] + 1) * 2.0**-24 * (size + abs(bias))
    if got.dtype == torch.bfloat16:
        bound = bound + 2.0**-8 * want.abs()
    assert bool(((got.double() - want).abs() <= bound).all())


# four parts: up to 4 rows, up to 96 x 16 columns; two: up to 8 rows, below 192 x 16; columns and rows that do
# not fill a workgroup's, steps of K that do not fill its waves, as few as one for all of them
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,K,parts", [(1, 1, 128, 4), (4, 1536, 640, 4), (3, 130, 1920, 4), (4, 1537, 128, 2), (5, 97, 64, 2),
                                         (8, 3055, 192, 2), (2, 2049, 2112, 2), (2, 2048, 2112, 2), (2, 2049, 1984, 2), (7, 1000, 7040, 2), (8, 3057, 128, 1),
                                         (9, 40, 256, 1)])
def test_parts_of_k(device, dtype, M, N, K, parts):
    g = torch.Generator(device=device).manual_seed(M * N + K)
    x, w = (torch.randn(n, K, device=device, generator=g).to(dtype) for n in (M, N))
    b = torch.randn(N, device=device, generator=g)
    out = torch.full((M + 1, N + 3), 7.0, dtype=dtype, device=device)  # (a row and columns past the result stay)
    tail = min(3, N - 1)
    t = torch.zeros(M, max(tail, 1), device=device)
    D.linear(x, w, out, M, bias=b, tail=(t, tail) if tail else None)
    if N > 2048 and K * out.element_size() > 4096:  # (a second round of workgroups over long rows)
        parts = 1
    label = native.last_variant()
    assert ("parts=%d" % parts in label) if parts > 1 else ("dense_gemv" in label and "parts" not in label), label
    check(out[:M, : N - tail], x, w[: N - tail], b[: N - tail].double())
    if tail:
        check(t, x, w[N - tail :], b[N - tail :].double())
    assert bool((out[M:] == 7).all()) and bool((out[:, N:] == 7).all())


# beyond one part's 192 x 16 columns: bytes of a row, and how full one part leaves its last round of 256 workgroups
@pytest.mark.parametrize("M,N,row,pair,parts", [
    (4, 3072, 1024, False, 2), (4, 4096, 2048, False, 1), (8, 5003, 2048, False, 2), (3, 16390, 2048, False, 1), (4, 8192, 4096, False, 2),
    (3, 16400, 3072, False, 1), (2, 16400, 3072, False, 2), (4, 5120, 6144, False, 2), (8, 5120, 6144, False, 1), (1, 6148, 8192, False, 2),
    (4, 4100, 13824, False, 2), (8, 4100, 13824, False, 1), (4, 3072, 3072, True, 1), (8, 4099, 3072, True, 2), (8, 4100, 13824, True, 2),
    (8, 7000, 2048, False, 1), (4, 12288, 16384, False, 1), (4, 5120, 16384, False, 2), (8, 6912, 4096, True, 1), (8, 4700, 4096, True, 2),
])
def test_parts_of_k_beyond_one_round(device, M, N, row, pair, parts):
    K = row // 2
    g = torch.Generator(device=device).manual_seed(M + N + K)
    x, w, u = (torch.randn(n, K, device=device, generator=g).bfloat16() for n in (M, N, N if pair else 1))
    out = torch.zeros(M, N, dtype=torch.bfloat16, device=device)
    if pair:  # (a gate of 1 and no bend: the product of the two)
        class Ones:
            limit, alpha, shift, cubic = float("inf"), 0.0, 0.0, 0.0

        D.glu(x, w, u, out, M, Ones)
    else:
        D.linear(x, w, out, M)
    assert ("parts=%d" % parts in native.last_variant()) if parts > 1 else "parts" not in native.last_variant(), native.last_variant()
    if not pair:
        check(out, x, w)
        return
    a, c = x.double() @ w.double().T, x.double() @ u.double().T  # sigmoid(0) = 1/2
    size_a, size_c = x.double().abs() @ w.double().abs().T, x.double().abs() @ u.double().abs().T
    bound = (K + 1) * 2.0**-24 * (size_a * c.abs() + size_c * a.abs()) * 0.51 + 2.0**-8 * (a * c / 2).abs()
    assert bool(((out.double() - a * c / 2).abs() <= bound + 1e-12).all())


# steps of K that are one batch of a wave's requests, one more, whole batches, and a last wave with none; where operands are requested
# in a ring and where not (9 rows; 5 rows in workgroups of 4 waves); two products of a launch with rows of different lengths
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,steps", [(1, 4096, 64), (4, 4100, 66), (8, 4096, 130), (9, 4100, 130), (5, 4099, 138), (3, 3500, 250), (4, 16400, 34), (5, 16385, 66),
                                       (1, 20, 66), (8, 2048, 132)])
def test_steps_of_a_wave(device, dtype, M, N, steps):
    size = dtype.itemsize
    K = (steps * 64 // size + 63) // 64 * 64
    g = torch.Generator(device=device).manual_seed(M + N + steps)
    x, w = (torch.randn(n, K, device=device, generator=g).to(dtype) for n in (M, N))
    out = torch.zeros(M, N, dtype=dtype, device=device)
    D.linear(x, w, out, M)
    assert "dense_gemv" in native.last_variant()
    check(out, x, w)
    x2, w2 = (torch.randn(n, K // 128 * 64, device=device, generator=g).to(dtype) for n in (M, 50))
    second = torch.zeros(M, 50, dtype=dtype, device=device)
    D.linear_pair(x, w, out, x2, w2, second, M)
    check(out, x, w)
    check(second, x2, w2)


# behind the norms of the residual: up to 128 x 16 columns always, below 256 x 16 with a float4 of a row per lane, beyond for rows of
# 4 KB; rows that are not whole vectors, columns that do not fill a workgroup's, steps that do not fill its waves
@pytest.mark.parametrize("dtype,M,N,H,two,pair,parts", [
    ("bf16", 1, 41, 70, True, False, 2), ("f32", 8, 2041, 250, False, True, 2), ("bf16", 2, 2048, 2000, True, True, 2), ("bf16", 3, 2048, 2000, True, True, 1), ("f32", 4, 2048, 512, False, False, 2),
    ("f32", 2, 3001, 1000, True, False, 2), ("f32", 2, 3001, 1000, False, True, 1), ("f32", 4, 3001, 1000, False, False, 1), ("bf16", 5, 2501, 320, False, False, 1),
    ("bf16", 2, 5001, 2048, False, False, 2), ("bf16", 1, 5001, 2048, True, False, 1), ("bf16", 1, 5700, 2048, False, False, 1), ("f32", 2, 9001, 1021, False, True, 2),
    ("bf16", 1, 2384, 2048, False, False, 2), ("f32", 2, 2273, 1000, False, False, 2),  # steps that fill half a batch: fewer columns than the product holds
    ("f32", 2, 4000, 4096, False, True, 1), ("f32", 2, 5000, 4096, False, True, 1), ("f32", 2, 6900, 4096, False, True, 1),  # 16 waves' sums and the rows: more than 64 KB of LDS
    # one batch of a wave, one and a part, two whole ones (requests in a ring) and more
    ("f32", 1, 9001, 1024, True, False, 1), ("f32", 1, 9001, 1500, False, False, 1), ("f32", 1, 9001, 2048, True, False, 1), ("bf16", 1, 16385, 2048, False, False, 1), ("f32", 1, 20001, 1030, True, False, 1),
])
def test_parts_of_k_behind_norms(device, dtype, M, N, H, two, pair, parts):
    dtype = torch.bfloat16 if dtype == "bf16" else torch.float32
    g = torch.Generator(device=device).manual_seed(M * N + H)
    rand = lambda *n: torch.randn(*n, device=device, generator=g)  # noqa: E731
    x, ld = rand(M, H), D.pad64(H)
    w, u = (torch.nn.functional.pad(rand(N, H), (0, ld - H)).to(dtype) for _ in range(2))
    br = D.Branches(rand(M, H), rand(H), 0.5, *((rand(M, H), rand(H), rand(H)) if two else ()))
    pre, xo, xb, op = rand(H), torch.zeros(M, H, device=device), torch.zeros(M, ld, dtype=dtype, device=device), torch.zeros(M, ld, dtype=dtype, device=device)
    out = torch.full((M + 1, N + 3), 7.0, dtype=dtype, device=device)

    class Ones:  # (a gate of 1 and no bend: half the product of the two)
        limit, alpha, shift, cubic = float("inf"), 0.0, 0.0, 0.0

    D.post_linear(x, br, 1e-5, xo, xb, w, out, M, pre=pre, up=u if pair else None, spec=Ones if pair else None)
    label = native.last_variant()
    assert "post" in label and ("parts=2" in label) == (parts == 2), label
    assert N not in (2384, 2273) or int(label.split("cols=")[1]) < 8, label
    D.post_norm_add(br, 1e-5, x, op, M, pre)
    # (sums of H squares in another order, up to three norms: less than 2 H roundings each; one more of the element type)
    near = 6 * H * 2.0**-24
    assert bool(((xo - x).abs() <= near * (x.abs() + 4)).all())
    off, size = (xb.float() - op.float()).abs(), op.float().abs()
    assert bool((off <= near * float(size.max()) + (2.0**-7 * size if dtype == torch.bfloat16 else 0)).all())
    assert not bool(xb[:, H:].any()) and bool((out[M:] == 7).all()) and bool((out[:, N:] == 7).all())
    got, w, u = out[:M, :N], w[:, :H], u[:, :H]
    if not pair:
        check(got, xb[:, :H], w)
        return
    o = xb[:, :H].double()
    a, c, size_a, size_c = o @ w.double().T, o @ u.double().T, o.abs() @ w.double().abs().T, o.abs() @ u.double().abs().T
    bound = (H + 1) * 2.0**-24 * (size_a * c.abs() + size_c * a.abs()) * 0.51 + (2.0**-8 if dtype == torch.bfloat16 else 2.0**-22) * (a * c / 2).abs()
    assert bool(((got.double() - a * c / 2).abs() <= bound + 1e-12).all())


# workgroups of fewer columns than a product holds, so that CUs get equal shares: one workgroup a CU and two, a last one of one column, the
# fewest of each number of parts, outputs whose last columns go to another buffer, a pair, two products, 4, 8 and 16 waves
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,K,kind", [(1, 2305, 4096, "plain"), (2, 6657, 2048, "plain"), (8, 6700, 2048, "plain"), (16, 2817, 3072, "plain"), (4, 6913, 2048, "pair"),
                                        (3, 1281, 1024, "pair"), (1, 766, 4096, "plain"), (9, 4353, 512, "pair"), (2, 2600, 2048, "dual"), (5, 6200, 3584, "dual")])
def test_columns_of_a_workgroup(device, dtype, M, N, K, kind):
    g = torch.Generator(device=device).manual_seed(M + N + K)
    x, w = (torch.randn(n, K, device=device, generator=g).to(dtype) for n in (M, N))
    out = torch.full((M + 1, N + 3), 7.0, dtype=dtype, device=device)
    if kind == "dual":
        n0, second = N // 3, torch.full((M + 1, N), 7.0, device=device)
        D.linear_pair(x, w[:n0], out, x, w[n0:], second, M)
        check(out[:M, :n0], x, w[:n0])
        check(second[:M, : N - n0], x, w[n0:])
        assert bool((out[:, n0:] == 7).all()) and bool((second[M:] == 7).all()) and bool((second[:, N - n0 :] == 7).all())
    elif kind == "pair":

        class Ones:  # (a gate of 1 and no bend: half the product of the two)
            limit, alpha, shift, cubic = float("inf"), 0.0, 0.0, 0.0

        u = torch.randn(N, K, device=device, generator=g).to(dtype)
        D.glu(x, w, u, out, M, Ones)
        a, c, size_a, size_c = (p.double() @ q.double().T for p, q in ((x, w), (x, u), (x.abs(), w.abs()), (x.abs(), u.abs())))
        bound = (K + 1) * 2.0**-24 * (size_a * c.abs() + size_c * a.abs()) * 0.51 + (2.0**-8 if dtype == torch.bfloat16 else 2.0**-22) * (a * c / 2).abs()
        assert bool(((out[:M, :N].double() - a * c / 2).abs() <= bound + 1e-12).all())
        assert bool((out[M:] == 7).all()) and bool((out[:, N:] == 7).all())
    else:
        t = torch.zeros(M, 37, device=device)
        D.linear(x, w, out, M, tail=(t, 37))
        check(out[:M, : N - 37], x, w[: N - 37])
        check(t, x, w[N - 37 :])
        assert bool((out[M:] == 7).all()) and bool((out[:, N - 37 :] == 7).all())
    label = native.last_variant()
    print(label)
    parts = int(label.split("parts=")[1].split()[0]) if "parts=" in label else 1
    cols = int(label.split("cols=")[1])
    assert 8 // parts <= cols < 16 // parts, label


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,K", [(1, 70, 128), (4, 1530, 896), (8, 2500, 192), (6, 2545, 320)])
def test_gated_pair_and_two_products(device, dtype, M, N, K):
    g = torch.Generator(device=device).manual_seed(M + N + K)
    x, x2, gate, up = (torch.randn(n, K, device=device, generator=g).to(dtype) * (1 if n == M else K**-0.5) for n in (M, M, N, N))

    class Plain:
        limit, alpha, shift, cubic = float("inf"), 1.0, 0.0, 0.0

    out = torch.zeros(M, N, dtype=torch.float32, device=device).to(dtype)
    D.glu(x, gate, up, out, M, Plain)
    assert "pair" in native.last_variant() and ("parts" in native.last_variant()) == (N <= 2544)
    a, c = x.double() @ gate.double().T, x.double() @ up.double().T
    want = a * torch.sigmoid(a) * c
    # (silu's slope stays below 1.1 and it below |a|; the two sums' errors as above, the gate's own work 2^-20)
    size_a, size_c = x.double().abs() @ gate.double().abs().T, x.double().abs() @ up.double().abs().T
    bound = (K + 1) * 2.0**-24 * (1.1 * size_a * c.abs() + size_c * a.abs()) * 1.01 + 2.0**-20 * want.abs()
    if dtype == torch.bfloat16:
        bound = bound + 2.0**-8 * want.abs()
    assert bool(((out.double() - want).abs() <= bound + 1e-12).all())

    n0 = N // 3
    y0, y1 = torch.zeros(M, n0, dtype=dtype, device=device), torch.zeros(M, N, dtype=torch.float32, device=device)
    D.linear_pair(x, gate[:n0].contiguous(), y0, x2, up, y1, M)
    assert "dual" in native.last_variant()
    check(y0, x, gate[:n0])
    check(y1, x2, up)


# the last columns of a GEMM of many rows in their float32 buffer: a whole block of 32 columns, part of one, none of
# the first buffer's block; rows that do not fill a tile
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,n1", [(17, 300, 256), (64, 300, 250), (65, 4100, 4000), (1000, 3300, 3232), (1000, 3300, 31), (770, 4097, 4096)])
def test_last_columns_of_a_gemm(device, dtype, M, N, n1):
    K = 128
    g = torch.Generator(device=device).manual_seed(M + N)
    x, w = torch.randn(M, K, device=device, generator=g).to(dtype), (torch.randn(N, K, device=device, generator=g) / 8).to(dtype)
    b = torch.randn(N, device=device, generator=g)
    out = torch.full((M + 1, n1 + 5), 7.0, dtype=dtype, device=device)
    t = torch.full((M + 1, N - n1 + 2), 7.0, device=device)
    D.linear(x, w, out, M, bias=b, tail=(t, N - n1))
    check(t[:M, : N - n1], x, w[n1:], b[n1:].double())
    check(out[:M, :n1], x, w[:n1], b[:n1].double())
    assert bool((out[M:] == 7).all()) and bool((out[:, n1:] == 7).all()) and bool((t[M:] == 7).all()) and bool((t[:, N - n1 :] == 7).all())


# K split over two workgroups per CU: from 24 steps of 64 per range where CUs are left over, from 48 where none is
@pytest.mark.parametrize("M,N,K,split", [(300, 2040, 6912, 4), (300, 2040, 5952, 2), (1000, 2048, 6144, 2), (1000, 2048, 6080, 1), (700, 2048, 3136, 2)])
def test_long_ranges_of_k(device, M, N, K, split):
    g = torch.Generator(device=device).manual_seed(K)
    x, w = (torch.randn(n, K, device=device, generator=g).bfloat16() for n in (M, N))
    out = torch.zeros(M, N, device=device)
    D.linear(x, w, out, M)
    assert native.last_variant().endswith("x%d" % split), native.last_variant()
    check(out, x, w)


@pytest.mark.parametrize("M,ldb,kind", [(4, 1 << 27, "tail"), (16, 1 << 26, "rows"), (4, 1 << 27, "factor"), (8, 3 << 25, "pair")])
def test_products_behind_branches_of_far_rows(device, M, ldb, kind):
    """Rows of a branch whose bytes do not fit 31 or 32 bits together: the same as rows that lie close."""
    H, N, T, two = 200, 96, 20, kind == "factor"
    g = torch.Generator(device=device).manual_seed(M)
    rand = lambda *n: torch.randn(*n, device=device, generator=g)  # noqa: E731
    x, gains, pre, bias, ld = rand(M, H), [rand(H) for _ in range(3)], rand(H), rand(N), D.pad64(H)
    w, u = (torch.nn.functional.pad(rand(N, H), (0, ld - H)).bfloat16() for _ in range(2))
    near = [rand(M, H) for _ in range(1 + two)]
    far = []
    for t in near:
        flat = torch.empty((M - 1) * ldb + H, device=device)
        far.append(flat.as_strided((M, H), (ldb, 1)).copy_(t))
    factor, rows = rand(M + 3, N).bfloat16(), torch.arange(M + 2, 2, -1, dtype=torch.int32, device=device)
    spec = SimpleNamespace(limit=7.0, alpha=1.702, shift=1.0, cubic=0.0)

    def run(b):
        br = D.Branches(b[0], gains[0], 0.5, *((b[1], gains[1], gains[2]) if two else ()))
        xo, xb = torch.empty(M, H, device=device), torch.zeros(M, ld, dtype=torch.bfloat16, device=device)
        out, tail = torch.full((M, N + 8), 7.0, dtype=torch.bfloat16, device=device), torch.full((M, T + 4), 7.0, device=device)
        kw = dict(tail=dict(bias=bias, tail=(tail, T)), rows=dict(after=D.After("relu2", mul=factor, rows=rows)),
                  factor=dict(after=D.After(mul=factor)), pair=dict(up=u, spec=spec))[kind]
        D.post_linear(x, br, 1e-5, xo, xb, w, out, M, pre=pre, **kw)
        return xo, xb.float(), out.float(), tail

    # the sums of a row over another number of waves: 2 H roundings for each of up to three norms; then, where that
    # turns a rounding to the operand's type, its last bit in some of the H products of a column
    (xo, *got), (xo_near, *want) = run(far), run(near)
    assert bool(((xo - xo_near).abs() <= 6 * H * 2.0**-24 * (xo_near.abs() + 4)).all())
    for a, b in zip(got, want):
        torch.testing.assert_close(a, b, rtol=2.0**-7, atol=2.0**-9 * float(b.abs().max()))


# rows of up to 256, 512 and 1024 threads' columns, full and not; columns past the row
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,H,two,gain,pre", [(1, 4, False, True, True), (3, 1000, True, True, False), (4, 1024, True, True, True), (2, 1028, False, False, True),
                                              (5, 2048, True, True, True), (4, 2052, False, True, False), (256, 3076, True, True, True), (2, 4096, False, False, False)])
def test_post_norm_of_few_rows(device, dtype, M, H, two, gain, pre):
    g = torch.Generator(device=device).manual_seed(M + H)
    r = lambda *n: torch.randn(*n, device=device, generator=g)  # noqa: E731
    x, a, b = r(M, H), r(M, H), r(M, H)
    ga, gb, gn, gp = (1 + 0.1 * r(H) for _ in range(4))
    unit = lambda v: v * (v.pow(2).mean(1, keepdim=True) + 1e-5).rsqrt()  # noqa: E731
    v = (unit(a.double()) * ga.double() + unit(b.double()) * gb.double()) / 2 if two else a.double()
    y = x.double() + 0.5 * (unit(v) * gn.double() if gain else v)
    ld = D.pad64(H)
    xb = torch.full((M + 1, ld), 7.0, dtype=dtype, device=device)
    D.post_norm_add(D.Branches(a, gn if gain else None, 0.5, *((b, ga, gb) if two else ())), 1e-5, x, xb, M, gp if pre else None)
    # a sum of H squares: a relative H / 4 + 10 roundings at most of 2^-24, halved by the root, three norms on end
    tol = 3 * (H / 4 + 20) * 2.0**-24
    assert bool(((x.double() - y).abs() <= tol * (y.abs() + v.abs().max() * 3)).all())
    want = unit(y) * gp.double() if pre else y
    assert bool(((xb[:M, :H].double() - want).abs() <= (tol + (2.0**-8 if dtype == torch.bfloat16 else 0)) * want.abs() + tol * want.abs().max()).all())
    assert bool((xb[M:] == 7).all()) and bool((xb[:, H:] == 7).all())


# parts of one team's columns in one pass and in two, and just beyond; a gain shorter than the row
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,size,groups,period", [(2, 64, 3, 64), (3, 256, 2, 512), (1, 516, 3, 516), (2, 1024, 3, 1024), (2, 1028, 2, 2056), (2, 2052, 1, 2052), (3, 45, 2, 45), (2, 4100, 1, 4100)])
def test_gated_norm_parts(device, dtype, M, size, groups, period):
    g = torch.Generator(device=device).manual_seed(size)
    W = size * groups
    y, z = (torch.randn(M, W, device=device, generator=g) for _ in range(2))
    z, gain = z.to(dtype), 1 + 0.1 * torch.randn(period, device=device, generator=g)
    for first in (True, False):
        out = torch.full((M, W + 4), 7.0, dtype=dtype, device=device)
        D.gated_norm(y, z, gain, out, M, W, groups, 1e-5, first)
        silu = z.double() * torch.sigmoid(z.double())
        v = (y.double() * silu if first else y.double()).view(M, groups, size)
        want = (v * (v.pow(2).mean(2, keepdim=True) + 1e-5).rsqrt()).view(M, W) * gain.double().repeat(W // period)
        want = want if first else want * silu
        tol = (size / 4 + 30) * 2.0**-24 + (2.0**-8 if dtype == torch.bfloat16 else 0)
        assert bool(((out[:, :W].double() - want).abs() <= tol * want.abs() + 1e-30).all())
        assert bool((out[:, W:] == 7).all())


# rows of up to 256, 512 and 1024 threads' columns, full and not, and beyond; a gain that does not begin at 16 bytes
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,H,center,at", [(1, 4, False, 0), (3, 1000, True, 0), (2, 1024, False, 0), (2, 1028, True, 0), (5, 2048, False, 1), (256, 2052, False, 0), (2, 4096, True, 0), (2, 4100, False, 0)])
def test_norm_of_few_rows(device, dtype, n, H, center, at):
    g = torch.Generator(device=device).manual_seed(n + H)
    x, gain = 1 + torch.randn(n + 2, H, device=device, generator=g), (1 + 0.1 * torch.randn(H + 4, device=device, generator=g))[at : at + H]
    rows = torch.randperm(n + 2, device=device, generator=g)[:n].int()
    out = torch.full((n + 1, H + 4), 7.0, dtype=dtype, device=device)
    D.norm_rows(x, gain, 1e-5, out, n, rows=rows, center=center)
    v = x[rows.long()].double()
    v = v - v.mean(1, keepdim=True) if center else v
    want = v * (v.pow(2).mean(1, keepdim=True) + 1e-5).rsqrt() * gain.double()
    # a mean's and a square sum's roundings, H / 4 + 10 each at most, of values up to some five times the root mean square
    tol = (H / 4 + 20) * 2.0**-24
    assert bool(((out[:n, :H].double() - want).abs() <= (tol + (2.0**-8 if dtype == torch.bfloat16 else 0)) * want.abs() + 5 * tol).all())
    assert bool((out[n:] == 7).all()) and bool((out[:, H:] == 7).all())


# gated pairs of few tiles: ranges of K and their sums in a launch of its own; a last range that is shorter, rows and columns that do not
# fill a tile, the most ranges (16), tiles of 64 rows and of 128, and pairs that stay whole.  split: in bf16, in float32
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,K,split,tall", [
    (17, 65, 1152, (True, True), False), (53, 2560, 1024, (True, True), False), (100, 333, 4800, (True, True), False), (64, 6912, 2048, (True, True), False),
    (129, 1990, 5952, (True, True), False), (700, 1100, 6016, (False, True), False), (17, 40, 8192, (True, True), False), (66, 16448, 8192, (True, True), True),
    (150, 8300, 4096, (False, True), True), (20, 400, 64, (False, False), False), (300, 7000, 256, (False, False), True)])
def test_gated_pair_in_ranges_of_k(device, dtype, M, N, K, split, tall):
    g = torch.Generator(device=device).manual_seed(M + N + K)
    x, gate, up = (torch.randn(n, K, device=device, generator=g).to(dtype) * (1 if n == M else K**-0.5) for n in (M, N, N))

    class Spec:
        limit, alpha, shift, cubic = 1.5, 1.702, 1.0, 0.0

    out = torch.full((M + 1, N + 5), 7.0, dtype=dtype, device=device)
    D.glu_gemm(x, gate, up, out, M, Spec)
    label = native.last_variant()
    assert "pair" in label and label.endswith("x1") != split[dtype == torch.float32], label
    assert "wide" in label or (",2,2,plain" in label) == tall, label
    assert K != 8192 or N > 40 or label.endswith("x16"), label
    a, c = x.double() @ gate.double().T, x.double() @ up.double().T
    want = a.clamp(max=1.5) * torch.sigmoid(1.702 * a.clamp(max=1.5)) * (c.clamp(-1.5, 1.5) + 1)
    # (the unit's slope stays below 1.1 and it below |a|; the two sums' errors as above, the unit's own work 2^-20, in bf16 2^-18, and a rounding)
    size_a, size_c = x.double().abs() @ gate.double().abs().T, x.double().abs() @ up.double().abs().T
    bound = (K + 1) * 2.0**-24 * (1.1 * size_a * 2.5 + size_c * 1.5) + (2.0**-20 if dtype == torch.float32 else 2.0**-8 + 2.0**-18) * want.abs()
    assert bool(((out[:M, :N].double() - want).abs() <= bound + 1e-12).all())
    assert bool((out[M:] == 7).all()) and bool((out[:, N:] == 7).all())


def test_gated_pairs_on_two_streams(device):
    """Pairs whose ranges of K meet in memory, on two streams side by side: each has the bits that it has alone."""
    M, N, K = 53, 2560, 1024
    g = torch.Generator(device=device).manual_seed(5)

    class Spec:
        limit, alpha, shift, cubic = 7.0, 1.702, 1.0, 0.0

    sets = [[torch.randn(n, K, device=device, generator=g) * K**-0.25 for n in (M, N, N)] for _ in range(2)]
    alone = [torch.empty(M, N, device=device) for _ in sets]
    for (x, gate, up), out in zip(sets, alone):
        D.glu(x, gate, up, out, M, Spec)
    assert "pair" in native.last_variant() and not native.last_variant().endswith("x1"), native.last_variant()
    outs = [[torch.empty(M, N, device=device) for _ in range(40)] for _ in sets]
    streams = [torch.cuda.Stream() for _ in sets]
    big = torch.randn(4096, 4096, device=device)
    for _ in range(6):  # (both queues fill up behind this)
        big = big @ big / 64
    behind = torch.cuda.Event()
    behind.record()
    for s in streams:
        s.wait_event(behind)
    for i in range(40):
        for (x, gate, up), out, s in zip(sets, outs, streams):
            with torch.cuda.stream(s):
                D.glu(x, gate, up, out[i], M, Spec)
    torch.cuda.synchronize()
    for want, out in zip(alone, outs):
        assert all(torch.equal(o, want) for o in out)


def test_gated_pair_of_more_rows_than_a_grid_holds(device):
    """A narrow pair of 65600 rows, whose sums' launch would be that many blocks high: whole, and in range at both ends."""
    M, N, K = 65600, 8, 1024
    g = torch.Generator(device=device).manual_seed(3)
    x, gate, up = (torch.randn(n, K, device=device, generator=g) * K**-0.25 for n in (M, N, N))

    class Spec:
        limit, alpha, shift, cubic = float("inf"), 0.0, 0.0, 0.0

    out = torch.full((M + 1, N), 7.0, device=device)
    D.glu(x, gate, up, out, M, Spec)
    assert native.last_variant().endswith("x1"), native.last_variant()
    for rows in (slice(0, 300), slice(M - 300, M)):  # (a gate of 1 and no bend: half the product of the two)
        a, c, size_a, size_c = (p.double() @ q.double().T for p, q in ((x[rows], gate), (x[rows], up), (x[rows].abs(), gate.abs()), (x[rows].abs(), up.abs())))
        bound = (K + 1) * 2.0**-24 * (size_a * c.abs() + size_c * a.abs()) * 0.51 + 2.0**-22 * (a * c / 2).abs()
        assert bool(((out[rows].double() - a * c / 2).abs() <= bound + 1e-12).all())
    assert bool((out[M:] == 7).all())
