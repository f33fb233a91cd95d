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


# one workgroup up to 256 keys of 128 or 512 of 64 (the matrix-core kernel, 16 and more pairs of 128: 256), several
# beyond; lengths differ inside a batch, and a second call finds the hand-over's counters as the first left them
@pytest.mark.parametrize("Hq,Hkv,D,S,lens", [
    (32, 8, 128, 4096, [1]), (32, 8, 128, 4096, [256]), (32, 8, 128, 4096, [257]), (32, 8, 64, 600, [512]), (32, 8, 64, 600, [513]),
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
