#!/usr/bin/env python3
"""Headline benchmark: batch-1 greedy decode of a Llama-3.1-8B-architecture model on MLX
4-bit g64 weights, one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W]

One "step" is one decoded token: the full shard forward (32 layers + head) as a HIP
graph replay at a context of about 2048 tokens, weights and KV cache resident in HBM,
greedy sampling on the device.  Prints ONE JSON line: decode tok/s (`value`), the
roofline of the dominant kernel (the fused dequant-GEMV, measured live with HIP events)
and the CPU oracle timed on this box's host cores (`cpu_baseline`, reported only).

Weights are synthetic (N(0,0.02) -> bf16 -> mx.quantize-style affine 4-bit g64), the
prompt is 2048 uniform random token ids; see `data` in the output.
"""

from __future__ import annotations

import argparse
import json
import os
import sys
import time

import numpy as np


# width, layers, heads, kv heads, head size, experts (identity ones among them), top, ff, vocab, bits of
# the Qwen3-MoE beside it
GEKAZEN_SIZES = {
    "1k": (1024, 24, 16, 8, 64, 64, 4, 4, 512, 65536, 4),
    "2k": (2048, 16, 32, 4, 128, 128, 8, 8, 768, 151936, 4),
    "4k": (4096, 6, 64, 4, 128, 128, 8, 8, 1536, 151936, 8),
}

# Novosun layers beside a Gekazen of that size: kinds of the layers (g linear attention, p attention beside a
# state-space recurrence), linear attention heads / key size / value size, recurrence heads / value size / state / groups, ff
NOVOSUN_SIZES = {
    "1k": ("gp" * 12, 4, 128, 256, 32, 64, 128, 1, 2560),
    "2k": ("gp" * 8, 4, 256, 512, 64, 64, 128, 1, 6912),
    "4k": ("gp" * 3, 8, 256, 512, 128, 64, 128, 8, 13824),
}

# Pimisun layers beside a Gekazen of that size (its attention and experts): kinds of the layers (l latent attention,
# a attention), latent heads / unrotated / rotated / value size / latent of queries / of keys and values, ff of the
# one dense layer, size of a token's vector
PIMISUN_SIZES = {
    "1k": ("la" * 12, 16, 64, 32, 64, 384, 256, 2560, 64),
    "2k": ("la" * 8, 16, 128, 64, 128, 1024, 512, 6912, 64),
    "4k": ("la" * 3, 64, 128, 64, 128, 1536, 512, 13824, 128),
}

# Zedotar layers beside a Novosun of that size (heads and head size of its attention, its feed-forward): kinds of the
# layers (w attention over a window with means of blocks behind it, s attention with sigmoid weights, m matrix
# memory), window, block, taps, memory heads / key size / value size
ZEDOTAR_SIZES = {
    "1k": ("wsm" * 8, 1024, 16, 4, 4, 128, 256),
    "2k": ("wsm" * 5 + "w", 1024, 16, 4, 4, 256, 512),
    "4k": ("wsm" * 2, 1024, 16, 4, 8, 256, 512),
}


def parse_args():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=128)
    ap.add_argument("--warmup", type=int, default=16)
    ap.add_argument("--config", default="llama-3.1-8b")
    ap.add_argument("--prompt", type=int, default=2048)
    ap.add_argument("--layers", type=int, default=None, help="debug: truncate the model")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--cpu-seconds", type=float, default=12.0)
    ap.add_argument("--no-graph", action="store_true")
    ap.add_argument("--no-engine", action="store_true", help="skip the run through the Engine")
    ap.add_argument("--batch", type=int, default=1, help="sequences decoded together (1..16)")
    ap.add_argument("--shard-layers", type=int, default=None,
                    help="run layers [0, n) as a first pipeline shard (output: hidden state)")
    ap.add_argument("--pmc-copy", action="store_true",
                    help="also launch one plain 256 MiB copy kernel: the known-size dispatch that "
                         "calibrates FETCH_SIZE / WRITE_SIZE in a rocprofv3 --pmc pass")
    ap.add_argument("--workload", default="decode", choices=["decode", "qmatmul_sweep", "gekazen", "novosun", "pimisun", "zedotar"],
                    help="decode (default, the headline), the quantised-matmul shape sweep, or a layer-list design "
                         "beside the closest other model of equal size, whole steps and launch by launch: Gekazen "
                         "beside a Qwen3-MoE, Novosun and Pimisun beside a Gekazen, Zedotar beside a Novosun")
    ap.add_argument("--gekazen-size", "--size", dest="size", default="all", choices=["all"] + list(GEKAZEN_SIZES),
                    help="sizes of the gekazen, novosun, pimisun and zedotar workloads")
    return ap.parse_args()


def qbytes(n: int, k: int, bits: int) -> int:
    return n * k * bits // 8 + n * (k // 64) * 4


def measure_kernels(model, torch, reps: int = 20):
    """Per-kernel HBM roofline of the GEMV launches of one decode step.  Each group of
    same-shaped launches (one per layer, distinct weights, 4.2 GB in total so nothing
    is served from cache) is captured into a HIP graph and timed with events on the
    launch stream; average launch duration = elapsed / launches."""
    from exo_amd import native, ops
    from exo_amd.model import capture_graph

    c = model.cfg
    dev = model.device
    H, D = c.hidden_size, c.head_dim
    Hq, Hkv, I = c.num_attention_heads, c.num_key_value_heads, c.intermediate_size
    bf = dict(dtype=torch.bfloat16, device=dev)
    xh = torch.randn(1, H, device=dev).to(torch.bfloat16)
    xa = torch.randn(1, Hq * D, device=dev).to(torch.bfloat16)
    xi = torch.randn(1, I, device=dev).to(torch.bfloat16)
    y_qkv = torch.empty(1, (Hq + 2 * Hkv) * D, **bf)
    y_h = torch.empty(1, H, **bf)
    y_i = torch.empty(1, I, **bf)
    y_v = torch.empty(1, c.vocab_size, **bf)
    def kernel_name():  # of the launch just made, from the instance that it reports
        return native.last_variant().split()[0].replace("<", "_kernel<", 1)

    nw, eps = torch.ones(H, **bf), c.rms_norm_eps

    def timed_rounds(graph, launches, rounds=5):
        """Average launch duration in us: `rounds` timed regions of `reps` replays each,
        the median region (the first one after a capture runs 2-3 % slow)."""
        avg = []
        for _ in range(rounds):
            st, en = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            st.record()
            for _ in range(reps):
                graph.replay()
            en.record()
            torch.cuda.synchronize()
            avg.append(st.elapsed_time(en) * 1e3 / (reps * launches))
        return sorted(avg)[len(avg) // 2]

    groups = {
        "norm_gate_up_swiglu": (lambda L: ops.qmv_swiglu(xh, L.gate, L.up, out=y_i, norm_weight=nw, eps=eps),
                                2 * qbytes(I, H, c.bits) + 2 * (2 * H + I)),
        "down_residual": (lambda L: ops.quantized_matmul(xi, L.down, residual=y_h, out=y_h),
                          qbytes(H, I, c.bits) + 2 * (I + 2 * H)),
        "norm_qkv": (lambda L: ops.quantized_matmul(xh, L.qkv, out=y_qkv, norm_weight=nw, eps=eps),
                     qbytes((Hq + 2 * Hkv) * D, H, c.bits) + 2 * (2 * H + (Hq + 2 * Hkv) * D)),
        "o_residual": (lambda L: ops.quantized_matmul(xa, L.o, residual=y_h, out=y_h),
                       qbytes(H, Hq * D, c.bits) + 2 * (Hq * D + 2 * H)),
    }
    out = []
    for name, (fn, nbytes) in groups.items():
        for L in model.layers:  # warm-up (also sets kernel attributes outside capture)
            fn(L)
        kname = kernel_name()
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with capture_graph(g):
            for L in model.layers:
                fn(L)
        g.replay()
        torch.cuda.synchronize()
        us = timed_rounds(g, len(model.layers))
        out.append(dict(name=name, kernel=kname, launches_per_token=len(model.layers),
                        bytes_per_launch=nbytes, avg_us=us, GBps=nbytes / us * 1e-3))
    # lm_head: once per token, with 4 GB of layer weights streamed since its last use, so
    # the 256 MB last-level cache holds none of it when it runs.  Re-reading ONE matrix back to
    # back would find most of it there (5.0 against 4.7 TB/s measured), so the launches of the
    # timed graph rotate over four copies of the matrix (1.2 GB).
    from exo_amd.ops import QuantizedWeight
    hd = model.lm_head
    heads = [hd] + [QuantizedWeight(hd.weight.clone(), hd.scales.clone(), hd.biases.clone(), hd.bits)
                    for _ in range(3)]
    for q in heads:
        ops.quantized_matmul(xh, q, out=y_v, norm_weight=nw, eps=eps)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with capture_graph(g):
        for q in heads:
            ops.quantized_matmul(xh, q, out=y_v, norm_weight=nw, eps=eps)
    g.replay()
    torch.cuda.synchronize()
    us = timed_rounds(g, len(heads))
    del heads
    nbytes = qbytes(c.vocab_size, H, c.bits) + 2 * (2 * H + c.vocab_size)
    out.append(dict(name="norm_lm_head", kernel=kernel_name(), launches_per_token=1,
                    bytes_per_launch=nbytes, avg_us=us, GBps=nbytes / us * 1e-3))
    return out


def cpu_baseline(model, torch, seconds: float, context: int):
    """The CPU oracle (C restatement of the quantised matmul + numpy ops) timed on this
    host: one decode token of the same architecture at the same context length.
    Bounded sample: 2 layers + head are run and the layer time is scaled to the full
    depth."""
    from oracle import cref
    from oracle import models as OM

    c = model.cfg
    n_sample = min(2, len(model.layers))

    def to_np(t):
        t = t.detach().cpu().contiguous()
        if t.dtype == torch.int32:
            return t.numpy().view(np.uint32)
        return t.view(torch.int16).numpy().view(np.uint16)

    w = {}

    def put(prefix, q):
        w[prefix + ".weight"], w[prefix + ".scales"], w[prefix + ".biases"] = (
            to_np(q.weight), to_np(q.scales), to_np(q.biases))

    Hq, Hkv, D = c.num_attention_heads, c.num_key_value_heads, c.head_dim
    for i in range(n_sample):
        L = model.layers[i]
        p = f"model.layers.{i}."
        nq, nk = Hq * D, Hkv * D
        put(p + "self_attn.q_proj", L.qkv[0:nq])
        put(p + "self_attn.k_proj", L.qkv[nq : nq + nk])
        put(p + "self_attn.v_proj", L.qkv[nq + nk : nq + 2 * nk])
        put(p + "self_attn.o_proj", L.o)
        put(p + "mlp.gate_proj", L.gate)
        put(p + "mlp.up_proj", L.up)
        put(p + "mlp.down_proj", L.down)
        w[p + "input_layernorm.weight"] = to_np(L.in_norm)
        w[p + "post_attention_layernorm.weight"] = to_np(L.post_norm)
    put("model.embed_tokens", model.embed_tokens)
    put("lm_head", model.lm_head)
    w["model.norm.weight"] = to_np(model.norm)
    ocfg = OM.Config(model_type=c.model_type, hidden_size=c.hidden_size, num_hidden_layers=n_sample,
                     num_attention_heads=Hq, num_key_value_heads=Hkv, head_dim=D,
                     intermediate_size=c.intermediate_size, vocab_size=c.vocab_size,
                     rms_norm_eps=c.rms_norm_eps, rope_theta=c.rope_theta, rope_scaling=c.rope_scaling,
                     tie_word_embeddings=False, group_size=64, bits=c.bits)
    om = OM.ShardModel(ocfg, w, use_c=True)
    rng = np.random.default_rng(0)
    cache = OM.make_kv_cache(n_sample)
    from oracle.affine import bf16_round

    for kv in cache:  # a context of `context` cached tokens (synthetic K/V)
        kv.k = bf16_round(rng.standard_normal((1, Hkv, context, D)).astype(np.float32))
        kv.v = bf16_round(rng.standard_normal((1, Hkv, context, D)).astype(np.float32))
        kv.offset = context
    tok = np.array([[1]])
    om(tok, cache)  # warm-up
    for kv in cache:
        kv.trim(1)
    t_full, n_full, t0 = 0.0, 0, time.perf_counter()
    while time.perf_counter() - t0 < seconds * 0.7 or n_full < 2:
        a = time.perf_counter()
        om(tok, cache)
        t_full += time.perf_counter() - a
        n_full += 1
        for kv in cache:
            kv.trim(1)
    x = bf16_round(rng.standard_normal((1, c.hidden_size)).astype(np.float32))
    t_head, n_head, t0 = 0.0, 0, time.perf_counter()
    while time.perf_counter() - t0 < seconds * 0.3 or n_head < 2:
        a = time.perf_counter()
        om.linear(x, "lm_head")
        t_head += time.perf_counter() - a
        n_head += 1
    t_full /= n_full
    t_head /= n_head
    t_layer = max(t_full - t_head, 1e-9) / n_sample
    t_token = t_layer * c.num_hidden_layers + t_head
    import importlib.util
    have = {m: importlib.util.find_spec(m) is not None for m in ("mlx", "mlx_lm")}
    mlx_note = ("mlx_lm: unavailable on this box (importlib finds neither mlx nor mlx_lm), so the baseline "
                "is this repository's own CPU restatement; " if not all(have.values()) else
                "mlx / mlx_lm are importable here but are not driven by this build; ")
    return dict(value=1.0 / t_token, unit="tok/s", cores=cref.num_threads(), kind="port",
                mlx_importable=have,
                sample=(mlx_note +
                        f"{n_full} decode steps of {n_sample} layers + lm_head at context {context} "
                        f"(layer {t_layer * 1e3:.1f} ms, head {t_head * 1e3:.1f} ms), layer time "
                        f"scaled to {c.num_hidden_layers} layers; oracle/qmm_ref.c with OpenMP + numpy"),
                host_cpus=os.cpu_count(), affinity=len(os.sched_getaffinity(0)))


PMC_SUMMARY = "profiles/decode_llama8b_4bit_bs1_pmc_traffic.md"


def pmc_traffic(launch: str):
    """HBM bytes per launch of one GEMV group as measured by the committed
    `rocprofv3 --pmc FETCH_SIZE` / `WRITE_SIZE` passes of this command (a text summary
    under profiles/; counters cannot be read from inside the process).  Returns (bytes,
    where the figure comes from) or (None, None): it is a recorded measurement of that
    earlier run, not of this one."""
    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), PMC_SUMMARY)
    val, commit = None, "unknown"
    try:
        with open(path) as fh:
            for line in fh:
                parts = line.split()
                if len(parts) == 3 and parts[0] == "traffic_bytes_per_launch" and parts[1] == launch:
                    val = int(parts[2])
                if len(parts) >= 2 and parts[0] == "measured_at_commit":
                    commit = parts[1]
    except OSError:
        pass
    if val is None:
        return None, None
    return val, f"{PMC_SUMMARY} (rocprofv3 --pmc passes recorded at commit {commit}; not re-measured by this run)"


def engine_rates(model, cfg, args, torch):
    """The same workload through the Engine the runner drives (BatchGenerator.step(): queue,
    prefill, double-buffered graph replays with device sampling, detokeniser, chunks):
    `generation_tps` as the reference defines it, (n-1)/(t_last - t_first) per request
    (src/exo/worker/engines/mlx/generator/batch_generate.py:418-426), summed over the
    requests of the batch; once greedy, once with the reference's default sampler
    (temperature 0.7, min-p 0.05)."""
    from exo_amd.engine import BatchGenerator
    from exo_amd.types import GenerationTask, TextGenerationTaskParams

    B, K = args.batch, args.steps + args.warmup
    eng = BatchGenerator(model=model, tokenizer=None, model_id=args.config,
                         max_seq=args.prompt + K + 72)
    g = torch.Generator().manual_seed(1234)
    prompts = [torch.randint(0, cfg.vocab_size, (args.prompt,), generator=g).tolist() for _ in range(B)]
    res = {}
    for label, temp in (("engine_tok_s", 0.0), ("engine_tok_s_sampled", 0.7)):
        for i, p in enumerate(prompts):
            eng.submit(GenerationTask(f"{label}-{i}", f"cmd-{i}", TextGenerationTaskParams(
                model=args.config, input=p, max_output_tokens=K, temperature=temp, bench=True)))
        tps, n_done = 0.0, 0
        while n_done < B:
            for _tid, ev in eng.step():
                st = getattr(ev, "stats", None)
                if st is not None:
                    tps += st.generation_tps
                    n_done += 1
        res[label] = tps
    res["engine_note"] = (f"{B} request(s) of {K} tokens through BatchGenerator.step(); generation_tps per "
                          "request as the reference defines it, summed")
    eng.close()
    return res


def active_token_bytes(model, cfg, ctx: int, batch: int) -> int:
    """Algorithmic HBM bytes of one decode step: every weight the step multiplies by (for
    MoE layers the router plus top-k experts per sequence, at most all experts) once,
    plus the K/V read of every sequence."""
    n = 0
    for L in model.layers:
        n += L.qkv.nbytes + L.o.nbytes
        if cfg.is_moe:
            per_expert = (L.gate.nbytes + L.up.nbytes + L.down.nbytes) // cfg.num_experts
            n += L.router.nbytes + per_expert * min(cfg.num_experts, cfg.num_experts_per_tok * batch)
        else:
            n += L.gate.nbytes + L.up.nbytes + L.down.nbytes
    if model.lm_head is not None:
        n += model.lm_head.nbytes
    kv = 2 * len(model.layers) * cfg.num_key_value_heads * cfg.head_dim * ctx * 2 * batch
    return n + kv


def qmatmul_sweep(args):
    """configs[1] of the baseline: y = x @ dq(W)^T over the listed (N, K), bits and M.
    Weight copies rotate so that nothing is served from cache; one HIP-graph replay holds
    one launch per copy; events on the launch stream give the average launch duration."""
    import torch

    from exo_amd import native, ops
    from exo_amd.model import capture_graph
    from exo_amd.ops import QuantizedWeight

    native.load()
    dev = torch.device("cuda:0")
    shapes = [(4096, 4096), (1024, 4096), (14336, 4096), (4096, 14336), (128256, 4096)]
    rows = []
    g = torch.Generator(device=dev).manual_seed(4321)
    for bits in (4, 8):
        for (N, K) in shapes:
            wbytes = qbytes(N, K, bits)
            copies = max(4, min(32, int(1.5e9 // wbytes) + 1))
            ws = []
            for _ in range(copies):
                w = torch.randint(-2**31, 2**31 - 1, (N, K * bits // 32), dtype=torch.int32, device=dev, generator=g)
                sc = (torch.rand(N, K // 64, device=dev, generator=g) * 0.01).bfloat16()
                bi = (torch.rand(N, K // 64, device=dev, generator=g) * -0.08).bfloat16()
                ws.append(QuantizedWeight(w, sc, bi, bits))
            for M in (1, 4, 16, 32, 64, 128, 2048):
                if M >= 128 and N * M * 2 > (1 << 30):
                    continue  # 128256 x 2048 outputs: not a shape the models produce
                x = torch.randn(M, K, device=dev, generator=g).bfloat16()
                y = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
                fns = [(lambda q=q: ops.quantized_matmul(x, q, out=y)) for q in ws]
                for f in fns:
                    f()
                torch.cuda.synchronize()
                gr = torch.cuda.CUDAGraph()
                with capture_graph(gr):
                    for f in fns:
                        f()
                gr.replay()
                torch.cuda.synchronize()
                reps = 10 if M <= 128 else 3
                st, en = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                st.record()
                for _ in range(reps):
                    gr.replay()
                en.record()
                torch.cuda.synchronize()
                us = st.elapsed_time(en) * 1e3 / (reps * copies)
                nbytes = wbytes + 2 * M * (K + N)
                flops = 2.0 * M * N * K
                rows.append(dict(bits=bits, N=N, K=K, M=M, us=round(us, 2), GBps=round(nbytes / us * 1e-3, 1),
                                 frac_hbm=round(nbytes / us * 1e-3 / 8000.0, 3),
                                 TFLOPs=round(flops / us * 1e-6, 1), frac_mfma=round(flops / us * 1e-6 / 2500.0, 3)))
                print(f"[sweep] b{bits} N={N} K={K} M={M}: {us:.1f} us", file=sys.stderr, flush=True)
            del ws
    best = max((r for r in rows if r["M"] == 1), key=lambda r: r["GBps"])
    dom = next(r for r in rows if (r["bits"], r["N"], r["K"], r["M"]) == (4, 14336, 4096, 1))
    print(json.dumps({
        "metric": "qmatmul HBM GB/s (% of 8 TB/s) over the shape sweep", "value": dom["GBps"], "unit": "GB/s",
        "n_gpus": 1, "steps": len(rows), "warmup": 1, "ms_per_step": dom["us"] * 1e-3,
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "bf16",
        "data": "synthetic",
        "config": {"workload": "configs[1]: quantised matmul sweep, bits {4,8} x 5 shapes x M {1,4,16,32,64,128,2048}; "
                               "value = 4-bit 14336x4096 at M=1"},
        "roofline": {"bound": "hbm", "achieved": dom["GBps"], "peak": 8000.0, "unit": "GB/s",
                     "frac": dom["GBps"] / 8000.0, "traffic": None},
        "best_M1": best, "rows": rows, "cpu_baseline": None}))


# ------------------------------------------------------------------ Gekazen beside Qwen3-MoE


def time_launches(torch, fns, reps: int = 10, rounds: int = 5) -> float:
    """Average us per launch group of `fns` (one per layer) as one captured graph: the median of
    `rounds` timed regions."""
    from exo_amd.model import capture_graph

    for f in fns:
        f()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with capture_graph(g):
        for f in fns:
            f()
    g.replay()
    torch.cuda.synchronize()
    avg = []
    for _ in range(rounds):
        st, en = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        st.record()
        for _ in range(reps):
            g.replay()
        en.record()
        torch.cuda.synchronize()
        avg.append(st.elapsed_time(en) * 1e3 / (reps * len(fns)))
    return sorted(avg)[len(avg) // 2]


def row_of(name, us, nbytes, flops):
    """A launch against its roofline: `x` = time over the longer of bytes / 8 TB/s and
    products / 2.5 PFLOP/s."""
    floor = max(nbytes / 8e6, flops / 2.5e9)
    return dict(launch=name, us=round(us, 2), MB=round(nbytes / 1e6, 3), GFLOP=round(flops / 1e9, 3),
                x=round(us / floor, 2) if floor else None)


def gekazen_model(torch, size, window):
    from exo_amd.stack_config import StackConfig, gekazen_dict
    from exo_amd.stack_model import StackModel

    H, n, hq, hkv, hd, E, ident, top, ff, V, _ = size
    cfg = StackConfig.from_dict(gekazen_dict(H, V, n, heads=hq, kv_heads=hkv, dim=hd, vdim=hd, experts=E - ident,
                                             identity=ident, top=top, ff=ff, shared_ff=ff, window=window))
    g = torch.Generator(device="cuda").manual_seed(0)

    class Random(dict):  # tensors drawn when the model asks for them
        def __missing__(self, key):
            f = key.split(".")
            shapes = {"embed": (V, H), "head": (V, H), "norm": (H,), "norm1": (H,), "norm2": (H,), "router": (E, H),
                      "correction": (E,), "sg": (1, H), "gate": (ff, H), "up": (ff, H), "down": (H, ff),
                      "q": (hq * hd, H), "k": (hkv * hd, H), "v": (hkv * hd, H), "o": (H, hq * hd)}
            shape = (shapes[f[-2]][0],) if f[-1] == "b" else shapes[f[-1]]
            std = 0.02 if len(shape) == 2 else 0.01
            return torch.empty(shape, dtype=torch.bfloat16, device="cuda").normal_(0.0, std, generator=g)

    return StackModel(cfg, Random())


def qwen_model(torch, size):
    from exo_amd.config import ModelConfig
    from exo_amd.model import ShardModel
    from exo_amd.synth import synth_weights

    H, n, hq, hkv, hd, E, _, top, ff, V, bits = size
    cfg = ModelConfig("qwen3_moe", H, n, hq, hkv, hd, 0, V, 1e-6, 1e6, None, False, 64, bits, E, top, ff, True)
    return ShardModel(cfg, synth_weights(cfg, seed=0, device="cuda:0"))


def launch_setup(torch, m, B, ctx):
    """Cache, buffers and batch of a step of B rows (B <= 16: single tokens at context ctx; else one prompt)."""
    cache = m.make_cache(1 if B > 16 else B, ctx + B + 64)
    g = torch.Generator().manual_seed(7)
    toks = lambda n: torch.randint(0, m.cfg.vocab_size, (n,), generator=g).tolist()  # noqa: E731
    if B > 16:
        cache.reserve([0], B)
        batch, bf = m._batch(cache, [(0, B)], []), m._buffers(1, B)
        bf.tokens[:B].copy_(torch.tensor(toks(B), dtype=torch.int32))
    else:
        for r in range(B):
            m.step(cache, [(r, toks(ctx), [])])
        bf = m._buffers(B, 1)
        bf.tokens.copy_(torch.tensor(toks(B), dtype=torch.int32))
        m.decode_step(cache, B, use_graph=False)
        from exo_amd.stack_model import _Batch
        batch = _Batch(B, torch.arange(B, dtype=torch.int32, device="cuda"), cache.pos[:B] - 1, m._keys_hint(cache, slice(0, B)))
    return cache, bf, batch


def expert_launches(torch, m, bf, B, Ls, picks, norm, add, rows, pre, product):
    """The launches of a mixture of experts over the layers Ls, with the experts ``picks`` that each chose."""
    from exo_amd import dense_ops as D
    from exo_amd import ops

    c, prompt, H = m.cfg, B > 16, m.cfg.hidden_size
    f = Ls[0].spec.mlp
    e, r = f.expert, f.router
    real = [int((p < r.experts).sum()) for p in picks]
    uniq = [len(set(p[p < r.experts].tolist())) for p in picks]
    pairs, experts = sum(real) / len(real), sum(uniq) / len(uniq)
    lg, idx, wt = bf.router_logits(Ls[0].ff.router.shape[0]), bf.idx(r.top), bf.wt(r.top)
    n = Ls[0].ff.router.shape[0]
    add(pre + "router", lambda L: product(L, L.ff.router, lg, L.ff.router_b, xb=bf.xb), 2 * n * H + 2 * B * (n + H), 2 * B * n * H)
    if prompt:
        add("routing", lambda L: D.moe_route(lg, L.ff.correction, r.scale, idx, wt, B, r.renorm), B * r.outputs * 4, 0)
    per = 2 * e.ff * H
    sh = f.shared.ff * H * 2
    if not prompt:
        for L in Ls:
            if (L.index, bf.cur) not in bf.experts:
                bf.experts[L.index, bf.cur] = D.ExpertRows(f, L.ff, bf, H, bf.h)
        ex = [bf.experts[L.index, bf.cur] for L in Ls]
        # every layer streams the experts it chose in the forward above
        logits = [torch.full((B, lg.shape[1]), -30.0, device="cuda").scatter_(1, p.long().to("cuda"), 3.0) for p in picks]
        set_logits = [(lambda t=t: lg[:B].copy_(t)) for t in logits]
        chosen = [p.to("cuda") for p in picks]
        set_idx = [(lambda t=t: idx[:B].copy_(t)) for t in chosen]
        both = lambda a, b: (lambda: (a(), b()))  # noqa: E731
        for name, pre_fns, fns, mats in (
                ("routing, experts: gate, up (+ shared)", set_logits, [(lambda x=x: x.glu(B)) for x in ex], 2),
                ("experts: down, weighted sum (+ shared)", set_idx, [(lambda x=x: x.down(B)) for x in ex], 1)):
            us = time_launches(torch, [both(a, b) for a, b in zip(pre_fns, fns)]) - time_launches(torch, pre_fns)
            rows.append(row_of(name, us, mats * (experts * per + sh), mats * 2 * (pairs * e.ff * H + B * f.shared.ff * H)))
    else:
        act, eo = bf.act(r.top, e.ff), bf.expert_out(r.top)
        bf.idx(r.top)[:B].copy_(picks[0].to("cuda"))
        ws = ops.moe_group(idx[:B], r.experts, check_indices=False)
        add("group", lambda L: ops.moe_group(idx[:B], r.experts, check_indices=False), B * r.top * 8, 0)
        add("experts: gate, up", lambda L: D.grouped_gemm(bf.xb, L.ff.gate, ws, act, B, r.top, up=L.ff.up, spec=e),
            2 * experts * per + 2 * B * H + 2 * pairs * e.ff, 4 * pairs * e.ff * H)
        add("experts: down", lambda L: D.grouped_gemm(act, L.ff.down, ws, eo, B, r.top, x_per_pair=True),
            experts * per + 2 * pairs * (H + e.ff), 2 * pairs * e.ff * H)
        sa, so = bf.shared_act(f.shared.ff), bf.shared_out()
        add("shared: gate, up", lambda L: D.glu_gemm(bf.xb, L.ff.s_gate, L.ff.s_up, sa, B, f.shared),
            2 * sh + 2 * B * (H + f.shared.ff), 4 * B * f.shared.ff * H)
        add("shared: down", lambda L: D.linear(sa, L.ff.s_down, so, B), sh + 2 * B * (H + f.shared.ff), 2 * B * f.shared.ff * H)
        add("expert sum, norm + residual", lambda L: D.moe_sum_post_norm(eo, idx, wt, so, lg, r.experts, L.ff.gate_col, L.norm2,
                                                                     c.eps, bf.h, bf.xb, B, norm=norm), 2 * (pairs + B) * H + 10 * B * H, 0)


def gekazen_launches(torch, m, B, ctx):
    """Per-launch times of a step of B rows (B <= 16: single tokens at context ctx; else one prompt)."""
    from exo_amd import dense_ops as D

    c, prompt = m.cfg, B > 16
    H, Ls = c.hidden_size, m.layers
    cache, bf, batch = launch_setup(torch, m, B, ctx)
    picks = []

    def hook(i, h):
        L = c.layers[i]
        picks.append(bf.idx(L.mlp.router.top)[:B].cpu())
    m.layer_hook = hook
    m._forward(cache, bf, batch, False)
    m.layer_hook = None
    a = c.layers[0].mixer
    att = [bound[0] for bound in m._mixers(cache)]
    qkv, out = bf.cols("proj", -(-Ls[0].n_main // 8) * 8), bf.mixed("attn", a.heads * a.vdim)
    vis = [min(i + 1, (a.window or 1 << 30) + a.keep_first) for i in (range(B) if prompt else [ctx] * B)]
    kvb = 2 * a.kv_heads * (a.dim + a.vdim) * (B if prompt else sum(vis))
    rows = []

    def add(name, fn, nbytes, flops):
        fns = [(lambda L=L: fn(L)) for L in Ls]
        rows.append(row_of(name, time_launches(torch, fns * -(-12 // len(fns))), nbytes, flops))

    def mm(n, k, extra=0):
        return 2 * n * k + 2 * B * (n + k) + extra, 2 * B * n * k
    nq = Ls[0].proj.shape[0]
    fused = not prompt and D.post_linear_fits(B, Ls[0].proj, bf.xb, H)  # norm + residual inside the next product
    other = torch.empty_like(bf.h)

    def product(L, w, out, bias=None, xb=None):
        if fused:
            D.post_linear(bf.h, D.Branches(bf.branch, L.norm1), c.eps, other, xb, w, out, B, bias)
        else:
            D.linear(bf.xb, w, out, B, bias=bias)
    pre = "norm, residual, " if fused else ""
    add(pre + "qkv + bias", lambda L: product(L, L.proj, qkv, L.proj_b), *mm(nq, H))
    if prompt:
        add("append keys, values", lambda L: att[L.index].append(qkv, batch.slot, batch.pos, B), 2 * kvb, 0)
        add("attention", lambda L: att[L.index].prompt(qkv, out, *batch.blocks[att[0].prompt_block(a)]),
            kvb + 4 * B * a.heads * a.dim, 2 * sum(vis) * a.heads * (a.dim + a.vdim))
    else:
        add("norm, append, attention", lambda L: att[L.index].rows(qkv, out, batch.slot, batch.pos, B, batch.keys, append=True),
            kvb, 2 * sum(vis) * a.heads * (a.dim + a.vdim))
    add("o + bias", lambda L: D.linear(out, L.parts[0].o, bf.branch, B, bias=L.parts[0].o_b), *mm(H, a.heads * a.vdim))
    if not fused:
        add("norm + residual (twice a layer)" if not prompt else "norm + residual",
            lambda L: D.post_norm_add(D.Branches(bf.branch, L.norm1), c.eps, bf.h, bf.xb, B), B * H * 14, 0)
    expert_launches(torch, m, bf, B, Ls, picks, c.norm, add, rows, pre, product)
    return rows


def qwen_launches(torch, m, B, ctx):
    from exo_amd import ops

    c, prompt = m.cfg, B > 16
    H, I, k, E = c.hidden_size, c.moe_intermediate_size, c.num_experts_per_tok, c.num_experts
    Hq, Hkv, Dh = c.num_attention_heads, c.num_key_value_heads, c.head_dim
    T = B if prompt else 1
    S = 1 if prompt else B
    cache = m.make_cache(S, ctx + B + 64)
    bf = m._buffers(S, T)
    bf.h.normal_()
    bf.n.normal_()
    bf.qkv.normal_()
    bf.attn.normal_()
    cache.offsets = [0 if prompt else ctx - 1] * S
    cache.sync_pos()
    hint, tab = m._keys_hint(cache, slice(0, S)), m._rope_table(cache.max_seq)
    wb = lambda q: q.nbytes if q.weight.dim() == 2 else q.nbytes // E  # noqa: E731
    L0, rows, eps = m.layers[0], [], c.rms_norm_eps
    kvb = 4 * Hkv * Dh * (B if prompt else B * ctx)
    keys = sum(range(1, B + 1)) if prompt else B * ctx

    def add(name, fn, nbytes, flops):
        rows.append(row_of(name, time_launches(torch, [(lambda i=i, L=L: fn(i, L)) for i, L in enumerate(m.layers)]), nbytes, flops))

    def lin(q, norm=None, res=None):
        return 2 * B * (q.N + q.K) + wb(q), 2 * B * q.N * q.K
    if not prompt:
        add("norm + qkv", lambda i, L: ops.quantized_matmul(bf.h, L.qkv, out=bf.qkv, norm_weight=L.in_norm, eps=eps), *lin(L0.qkv))
        add("rope, norm, append, attention", lambda i, L: ops.attn_decode(
            bf.qkv, cache.k[i], cache.v[i], cache.pos, m.inv_freq, bf.attn, bf.sdpa_ws, m.scale, B, Hq, Hkv, Dh, L.q_norm,
            L.k_norm, eps, rope_tab=tab, keys_hint=hint), kvb, 4 * keys * Hq * Dh)
        add("o + residual", lambda i, L: ops.quantized_matmul(bf.attn, L.o, residual=bf.h, out=bf.h), *lin(L0.o))
        add("norm + router", lambda i, L: ops.quantized_matmul(bf.h, L.router, out=bf.router_logits, norm_weight=L.post_norm, eps=eps), *lin(L0.router))
        bf.router_logits.normal_()
        idx, sc, _ = ops.route_gather_qmv_swiglu(bf.h, bf.router_logits, k, True, L0.gate, L0.up, out=bf.act, norm_weight=L0.post_norm, eps=eps)
        uniq = len(set(idx.flatten().tolist()))
        add("routing, norm, experts: gate, up", lambda i, L: ops.route_gather_qmv_swiglu(
            bf.h, bf.router_logits, k, True, L.gate, L.up, out=bf.act, norm_weight=L.post_norm, eps=eps),
            2 * uniq * wb(L0.gate), 4 * B * k * I * H)
        add("experts: down, sum + residual", lambda i, L: ops.gather_qmv_combine(
            bf.act, L.down, idx, sc, residual=bf.h, out=bf.h, scratch=bf.expert_out, check_indices=False),
            uniq * wb(L0.down), 2 * B * k * I * H)
        return rows
    add("norm", lambda i, L: ops.rms_norm(bf.h, L.in_norm, eps, out=bf.n), 4 * B * H, 0)
    add("qkv", lambda i, L: ops.quantized_matmul(bf.n, L.qkv, out=bf.qkv), *lin(L0.qkv))
    add("rope, append", lambda i, L: ops.rope_kv_append(bf.qkv, bf.q, cache.k[i], cache.v[i], cache.pos, m.inv_freq, 1, B, Hq, Hkv, Dh,
                                                        L.q_norm, L.k_norm, eps, rope_tab=tab), 4 * B * (Hq + 2 * Hkv) * Dh, 0)
    add("attention", lambda i, L: ops.sdpa_prefill(bf.q, cache.k[i], cache.v[i], cache.pos, bf.attn, m.scale, 1, B, Hq, Hkv, Dh),
        kvb + 4 * B * Hq * Dh, 4 * keys * Hq * Dh)
    add("o + residual", lambda i, L: ops.quantized_matmul(bf.attn, L.o, residual=bf.h, out=bf.h), *lin(L0.o))
    add("router", lambda i, L: ops.quantized_matmul(bf.n, L.router, out=bf.router_logits), *lin(L0.router))
    bf.router_logits.normal_()
    add("routing", lambda i, L: ops.router_topk(bf.router_logits, k, True), 2 * B * E, 0)
    idx, sc = ops.router_topk(bf.router_logits, k, True)
    ws = ops.moe_group(idx, E, check_indices=False)
    add("group", lambda i, L: ops.moe_group(idx, E, check_indices=False), B * k * 8, 0)
    add("experts: gate, up", lambda i, L: ops.grouped_qmm_swiglu(bf.n.view(B, 1, -1), L.gate, L.up, ws, k, out=bf.act),
        2 * E * wb(L0.gate) + 2 * B * H + 2 * B * k * I, 4 * B * k * I * H)
    add("experts: down", lambda i, L: ops.grouped_qmm(bf.act, L.down, ws, k, out=bf.expert_out), E * wb(L0.down) + 2 * B * k * (I + H), 2 * B * k * I * H)
    add("expert sum + residual", lambda i, L: ops.moe_combine(bf.expert_out, sc, residual=bf.h, out=bf.h), 2 * B * (k + 2) * H, 0)
    return rows


class RandomTensors(dict):
    """Tensors of a layer-list checkpoint, drawn when the model asks for them; ``shape_of``: name -> shape."""

    def __init__(self, torch, shape_of):
        super().__init__()
        self.torch, self.shape_of = torch, shape_of
        self.g = torch.Generator(device="cuda").manual_seed(0)

    def __missing__(self, key):
        shape, mean, std = self.shape_of(key)
        t = self.torch.empty(shape, dtype=self.torch.bfloat16, device="cuda").normal_(0.0, std, generator=self.g)
        return t.add_(mean)


def novosun_model(torch, size, novo):
    from exo_amd.stack_config import StackConfig, novosun_dict
    from exo_amd.stack_model import StackModel

    H, _, hq, hkv, hd, _, _, _, _, V, _ = size
    kinds, lh, ld, lv, sh, sv, sn, sg, ff = novo
    cfg = StackConfig.from_dict(novosun_dict(H, V, kinds, heads=hq, kv_heads=hkv, dim=hd, vdim=hd, ff=ff, lin_heads=lh,
                                             lin_dim=ld, lin_vdim=lv, ssm_heads=sh, ssm_vdim=sv, ssm_state=sn,
                                             ssm_groups=sg, mult=0.5))
    inner, rank = sh * sv, 16
    ch = inner + 2 * sg * sn
    vectors = {"norm1": H, "norm2": H, "norm1b": H, "norm2b": H, "left.out": H, "right.out": H, "final.norm": H, "q.norm": hd,
               "k.norm": hd, "right.norm": inner, "mix.norm": lv, "A_log": sh, "D": sh}
    mats = {"embed": (V, H), "head": (V, H), "mlp.gate": (ff, H), "mlp.up": (ff, H), "mlp.down": (H, ff),
            "left.q": (hq * hd, H), "left.k": (hkv * hd, H), "left.v": (hkv * hd, H), "left.g": (hq, H), "left.o": (H, hq * hd),
            "right.in": (inner + ch + sh, H), "right.conv": (ch, 4), "right.o": (H, inner), "mix.q": (lh * ld, H),
            "mix.k": (lh * ld, H), "mix.v": (lh * lv, H), "mix.g": (lh * lv, H), "mix.o": (H, lh * lv), "mix.a1": (rank, H),
            "mix.a2": (lh * ld, rank)}

    def shape_of(key):
        for name, n in vectors.items():
            if key == name or key.endswith("." + name):
                return (n,), 1.0, 0.1
        for name, n in (("a2.b", lh * ld), ("conv.b", ch), ("dt_bias", sh)):
            if key.endswith(name):
                return (n,), {"a2.b": 2.0, "conv.b": 0.0, "dt_bias": -3.0}[name], 0.5
        for name, shape in mats.items():
            if key == name or key.endswith("." + name):
                return shape, 0.0, 0.3 if name in ("right.conv", "mix.a2") else 0.02
        raise KeyError(key)

    w = RandomTensors(torch, shape_of)
    for i, k in enumerate(kinds):  # (its size says the rank)
        if k == "g":
            w[f"l{i}.mix.a1"] = w[f"l{i}.mix.a1"]
    return StackModel(cfg, w)


def novosun_launches(torch, m, B, ctx):
    """Per-launch times of a step of B rows (B <= 16: single tokens at context ctx; else one prompt)."""
    from exo_amd import dense_ops as D
    from exo_amd.stack_layers import LinearAttentionPart

    c, prompt = m.cfg, B > 16
    H, eps = c.hidden_size, c.eps
    cache, bf, batch = launch_setup(torch, m, B, ctx)
    m._forward(cache, bf, batch, False)
    lin = [(L, o) for L, o in zip(m.layers, m._mixers(cache)) if isinstance(L.parts[0], LinearAttentionPart)]
    par = [(L, o) for L, o in zip(m.layers, m._mixers(cache)) if len(L.parts) > 1]
    every = [(L, None) for L in m.layers]
    rows, fused = [], not prompt and D.post_linear_fits(B, m.layers[0].proj, bf.xb, H, True)
    other = torch.empty_like(bf.h)

    def add(name, which, fn, nbytes, flops):
        fns = [(lambda L=L, o=o: fn(L, o)) for L, o in which]
        rows.append(row_of(name, time_launches(torch, fns * -(-12 // len(fns))), nbytes, flops))

    def mm(n, k):
        return 2 * n * k + 2 * B * (n + k), 2 * B * n * k

    def due(L, two):
        return D.Branches(bf.branch, L.norm1, c.norm.mult, *((bf.branch2, L.gain_a, L.gain_b) if two else ()))

    def product(L, w, out, two=False, **kw):
        pre = L.pre2 if "up" in kw else L.pre1
        if fused:
            D.post_linear(bf.h, due(L, two), eps, other, None, w, out, B, pre=pre, **kw)
        elif "up" in kw:
            D.glu(bf.xb, w, kw["up"], out, B, kw["spec"])
        else:
            D.linear(bf.xb, w, out, B, **kw)
    head = "norms, residual, " if fused else ""
    for name, which in (("linear attention", lin), ("attention | state space", par)):
        L0 = which[0][0]
        y = bf.cols("proj", -(-L0.n_main // 8) * 8)
        y2 = bf.f32("proj_tail", L0.n_tail)
        add(f"{head}{name}: projection", which, lambda L, o: product(L, L.proj, y, tail=(y2, L.n_tail)), *mm(L0.proj.shape[0], H))
        for i, p in enumerate(L0.parts):
            s = p.spec
            if hasattr(s, "kv_heads"):
                vis = [j + 1 for j in range(B)] if prompt else [ctx] * B
                kvb = 2 * s.kv_heads * (s.dim + s.vdim) * (B if prompt else sum(vis))
                fl = 2 * sum(vis) * s.heads * (s.dim + s.vdim)
                out = bf.mixed("attn", p.width)
                gate = y2[:, p.tcol :]
                if prompt:
                    add("append keys, values", which, lambda L, o: o[i].append(y[:, p.col :], batch.slot, batch.pos, B), 2 * kvb, 0)
                    add("attention", which, lambda L, o: o[i].prompt(y[:, p.col :], out, *batch.blocks[o[i].prompt_block(s)], gate=gate),
                        kvb + 4 * B * s.heads * s.dim, fl)
                else:
                    add("norm, append, attention", which, lambda L, o: o[i].rows(y[:, p.col :], out, batch.slot, batch.pos, B, batch.keys,
                                                                                append=True, gate=gate), kvb, fl)
                continue
            h, grp, d, e = s.core
            ins = 2 * (s.channels if hasattr(s, "channels") else h * (2 * d + e))
            part = "state space" if hasattr(s, "channels") else "linear attention"
            state = 8 * h * d * e * (1 if prompt else B)
            # at least: inputs and outputs once, the state in and out; two products with it per token
            add(f"{part}: recurrence", which, lambda L, o: L.parts[i]._recur(o[i], bf, batch, h * d if part[0] == "l" else h, part[0] == "s"),
                B * (ins + 4 * h * e) + state, 4 * B * h * d * e)
            z = y[:, p.col :] if part[0] == "s" else y[:, p.col + 2 * h * d + h * e :]
            ro, oo = bf.f32("recur", h * e), bf.mixed("recur_out", h * e)
            add(f"{part}: gated norm", which, lambda L, o: D.gated_norm(ro, z, L.parts[i].norm, oo, B, h * e, s.norm_groups if part[0] == "s" else h,
                                                                       eps, part[0] == "s"), B * h * e * 8, 0)
        if len(L0.parts) == 1:
            add(f"{name}: o", which, lambda L, o: D.linear(bf.mixed("recur_out", L.parts[0].width), L.parts[0].o, bf.branch, B),
                *mm(H, L0.parts[0].width))
        else:
            a, b = L0.parts[0].width, L0.parts[1].width
            nb, fl = mm(H, a + b)
            add(f"{name}: both o", which, lambda L, o: D.linear_pair(bf.mixed("attn", a), L.parts[0].o, bf.branch, bf.mixed("recur_out", b),
                                                                    L.parts[1].o, bf.branch2, B), nb, fl)
    if not fused:
        add("norms + residual", lin, lambda L, o: D.post_norm_add(due(L, False), eps, bf.h, bf.xb, B, L.pre2), B * H * 14, 0)
        add("norms of two branches + residual", par, lambda L, o: D.post_norm_add(due(L, True), eps, bf.h, bf.xb, B, L.pre2), B * H * 18, 0)
    f = c.layers[0].mlp
    act = bf.mixed("ff", f.ff)
    add(f"{head}gate, up", every, lambda L, o: product(L, L.ff.gate, act, len(L.parts) > 1, up=L.ff.up, spec=f), *mm(2 * f.ff, H))
    add("down", every, lambda L, o: D.linear(act, L.ff.down, bf.branch, B), *mm(H, f.ff))
    return rows


def pimisun_model(torch, size, pimi):
    from exo_amd.stack_config import StackConfig, pimisun_dict
    from exo_amd.stack_model import StackModel

    H, _, hq, hkv, hd, E, ident, top, eff, V, _ = size
    kinds, lh, ld, lr, lv, qr, kr, ff, side = pimi
    E -= ident
    cfg = StackConfig.from_dict(pimisun_dict(H, V, kinds, heads=hq, kv_heads=hkv, dim=hd, rot=hd // 2, window=4096, lat_heads=lh,
                                             lat_dim=ld, lat_rot=lr, lat_vdim=lv, q_rank=qr, kv_rank=kr, ff=ff, experts=E, top=top,
                                             expert_ff=eff, shared_ff=eff, side=side))
    vectors = {"norm1": H, "norm2": H, "final.norm": H, "side.norm": H, "q.norm": hq * hd, "k.norm": hkv * hd, "dq.norm": qr,
               "dkv.norm": kr, "router.b": E}
    mats = {"side.embed": (V, len(kinds) * side), "side.gate": (side, H), "side.proj": (H, side), "embed": (V, H), "mix.q": (hq * hd, H),
            "mix.k": (hkv * hd, H), "mix.v": (hkv * hd, H), "mix.dq": (qr, H), "mix.uq": (lh * (ld + lr), qr), "mix.dkv": (kr + lr, H),
            "mix.uk": (lh * ld, kr), "mix.uv": (lh * lv, kr), "mlp.router": (E, H), "mlp.up": (ff, H), "mlp.down": (H, ff)}

    def shape_of(key):
        for name, n in vectors.items():
            if key == name or key.endswith("." + name):
                return (n,), 0.0 if name == "router.b" else 1.0, 0.1
        if key.endswith("vmix"):
            return (), 0.4, 0.1
        if key.endswith("mix.o"):
            i = int(key[1 : key.index(".")])
            return (H, lh * lv if kinds[i] == "l" else hq * hd), 0.0, 0.02
        for name, shape in mats.items():
            if key == name or key.endswith("." + name):
                return shape, 0.0, 0.02
        return (H, eff) if key.endswith("down") else (eff, H), 0.0, 0.02  # an expert's

    return StackModel(cfg, RandomTensors(torch, shape_of))


def pimisun_launches(torch, m, B, ctx):
    """Per-launch times of a step of B rows (B <= 16: single tokens at context ctx; else one prompt)."""
    from exo_amd import dense_ops as D
    from exo_amd.stack_config import LatentSpec, MoeSpec

    c, prompt = m.cfg, B > 16
    H, eps = c.hidden_size, c.eps
    cache, bf, batch = launch_setup(torch, m, B, ctx)
    picks = []

    def hook(i, h):
        if isinstance(c.layers[i].mlp, MoeSpec):
            picks.append(bf.idx(c.layers[i].mlp.router.top)[:B].cpu())
    m.layer_hook = hook
    m._forward(cache, bf, batch, False)
    m.layer_hook = None
    op = [bound[0] for bound in m._mixers(cache)]
    every = m.layers
    lat, att = ([L for L in every if isinstance(L.spec.mixer, LatentSpec) == t] for t in (True, False))
    moe, dense = ([L for L in every if isinstance(L.spec.mlp, MoeSpec) == t] for t in (True, False))
    rows, fused = [], not prompt and D.post_linear_fits(B, every[0].proj, bf.xb, H)
    other = torch.empty_like(bf.h)

    def add(name, fn, nbytes, flops, which=moe):
        fns = [(lambda L=L: fn(L)) for L in which]
        rows.append(row_of(name, time_launches(torch, fns * -(-12 // len(fns))), nbytes, flops))

    def mm(n, k, rows=B):
        return 2 * n * k + 2 * rows * (n + k), 2 * rows * n * k

    def product(L, w, out, bias=None, xb=None, after=None):
        if fused:
            D.post_linear(bf.h, D.Branches(bf.branch, L.norm1, norm=c.norm), eps, other, xb, w, out, B, bias, after=after)
        else:
            D.linear(bf.xb, w, out, B, bias=bias, after=after)
    pre = "norm, residual, " if fused else ""
    # attention
    a, L0 = att[0].spec.mixer, att[0]
    qkv, out = bf.cols("proj", -(-L0.n_main // 8) * 8), bf.mixed("attn", a.heads * a.vdim)
    vis = [min(i + 1, a.window or 1 << 30) for i in (range(B) if prompt else [ctx] * B)]
    kvb = 2 * a.kv_heads * (a.dim + a.vdim) * (B if prompt else sum(vis))
    add(pre + "qkv", lambda L: product(L, L.proj, qkv), *mm(L0.n_main, H), att)
    fl = 2 * sum(vis) * a.heads * (a.dim + a.vdim)
    if prompt:
        add("norm, turn queries; append keys, values", lambda L: op[L.index].append(qkv, batch.slot, batch.pos, B),
            2 * kvb + 4 * B * a.heads * a.dim, 0, att)
        add("attention", lambda L: op[L.index].prompt(qkv, out, *batch.blocks[op[L0.index].prompt_block(a)]),
            kvb + 4 * B * a.heads * a.dim, fl, att)
    else:
        add("norm, append, attention", lambda L: op[L.index].rows(qkv, out, batch.slot, batch.pos, B, batch.keys, append=True), kvb, fl, att)
    add("o", lambda L: D.linear(out, L.parts[0].o, bf.branch, B), *mm(H, a.heads * a.vdim), att)
    # latent attention
    s, L0 = lat[0].spec.mixer, lat[0]
    p, n = L0.parts[0], s.heads
    down = bf.f32("proj_tail", -(-L0.n_tail // 8) * 8)
    q, lo = bf.mixed("lat_q", p.q_cols), bf.mixed("attn", p.width)
    ql, ol, lc = *(bf.mixed(x, n * D.pad64(s.kv_rank)) for x in ("lat_ql", "lat_ol")), bf.mixed("lat_c", s.q_rank)
    keys = [i + 1 for i in range(B)] if prompt else [ctx] * B
    store = 2 * (s.kv_rank + s.rot_dim) * (B if prompt else sum(keys))
    add(pre + "latent: down projections", lambda L: product(L, L.proj, down), *mm(L0.n_tail, H), lat)
    kv = down[:, s.q_rank :]
    add("latent: norm, queries", lambda L: D.norm_linear(down, L.parts[0].q_gain, eps, lc, L.parts[0].uq, q, B),
        *mm(n * (s.dim + s.rot_dim), s.q_rank), lat)
    if prompt:
        add("latent: norm, turn, append", lambda L: op[L.index].prepare(q, kv, batch.slot, batch.pos, B),
            B * (6 * (s.kv_rank + s.rot_dim) + 4 * n * s.rot_dim), 0, lat)
        parts = {L.index: dict(op[L.index].prompt_launches(q, kv, lo, batch.slot, batch.pos, *batch.latent.lists)) for L in lat}
        dk = s.dim + s.rot_dim
        for name, nb, g in (("gather", 2 * store, 0), ("keys", *mm(n * s.dim, s.kv_rank)), ("values", *mm(n * s.vdim, s.kv_rank)),
                            ("attention", 2 * B * n * 2 * (dk + s.vdim), 2 * sum(keys) * n * (dk + s.vdim))):
            add(f"latent: {name}", lambda L: parts[L.index][name](), nb, g, lat)
    else:
        add("latent: keys into queries, attention, values", lambda L: op[L.index].rows(q, kv, ql, ol, lo, batch.slot, batch.pos, B, batch.keys,
                                                                                      append=True),
            store + 2 * n * s.kv_rank * (s.dim + s.vdim), 2 * sum(keys) * n * (2 * s.kv_rank + s.rot_dim), lat)
        add("latent: - keys into queries", lambda L: D.head_linear(q, p.nope_pad, L.parts[0].uk, ql, D.pad64(s.kv_rank), B, s.dim),
            *mm(n * s.kv_rank, s.dim), lat)
        add("latent: - values (no merge)", lambda L: D.head_linear(ol, D.pad64(s.kv_rank), L.parts[0].uv, lo, s.vdim, B, s.kv_rank),
            *mm(n * s.vdim, s.kv_rank), lat)
    add("latent: o", lambda L: D.linear(lo, L.parts[0].o, bf.branch, B), *mm(H, p.width), lat)
    # feed-forwards, the tokens' vectors
    if not fused:
        add("norm of the sum", lambda L: D.post_norm_add(D.Branches(bf.branch, L.norm1, norm=c.norm), eps, bf.h, bf.xb, B), B * H * 14, 0, every)
    f = dense[0].spec.mlp
    act = bf.mixed("ff", f.ff)
    add(pre + "dense: up, square of relu", lambda L: product(L, L.ff.up, act, after=L.ff.after), *mm(f.ff, H), dense)
    add("dense: down", lambda L: D.linear(act, L.ff.down, bf.branch, B), *mm(H, f.ff), dense)
    expert_launches(torch, m, bf, B, moe, picks, c.norm, add, rows, pre, product)
    sa = bf.mixed("side", c.side_dim)
    add(pre + "token vector: gate", lambda L: product(L, L.side.gate, sa, after=D.After("gelu_tanh", L.side.table, bf.tokens)),
        *mm(c.side_dim, H), every)
    add("token vector: projection", lambda L: D.linear(sa, L.side.proj, bf.branch, B), *mm(H, c.side_dim), every)
    return rows


def zedotar_model(torch, size, novo, zedo):
    from exo_amd.stack_config import StackConfig, zedotar_dict
    from exo_amd.stack_model import StackModel

    H, _, hq, hkv, hd, _, _, _, _, V, _ = size
    kinds, win, pool, taps, mh, md, mv = zedo
    ff = novo[-1]
    cfg = StackConfig.from_dict(zedotar_dict(H, V, kinds, heads=hq, kv_heads=hkv, dim=hd, vdim=hd, rot=hd // 2, window=win, pool=pool,
                                             sig_heads=hq, sig_kv_heads=hkv, sig_dim=hd, sig_rot=hd, conv=taps, mem_heads=mh,
                                             mem_dim=md, mem_vdim=mv, ff=ff))
    q, kv, mk, me = hq * hd, hkv * hd, mh * md, mh * mv
    own = {"w": {"q": (q, H), "k": (kv, H), "v": (kv, H), "q.b": (q,), "k.b": (kv,), "v.b": (kv,), "g": (hq, H), "o": (H, q)},
           "s": {"q": (q, H), "k": (kv, H), "q.b": (q,), "k.b": (kv,), "q.conv": (q, taps), "k.conv": (kv, taps), "pb": (hq,),
                 "g": (q, H), "o": (H, q)},
           "m": {"q": (mk, H), "k": (mk, H), "v": (me, H), "g": (me, H), "i": (mh, H), "f": (mh, H), "i.b": (mh,), "f.b": (mh,),
                 "norm": (me,), "o": (H, me)}}
    mats = {"embed": (V, H), "head": (V, H), "mlp.gate": (ff, H), "mlp.up": (ff, H), "mlp.down": (H, ff)}
    means = {"pb": -6.0, "f.b": 4.0, "norm": 1.0}

    def shape_of(key):
        layer, _, name = key.partition(".")
        if key in mats or name in mats:
            return mats.get(key) or mats[name], 0.0, 0.02
        if not name.startswith("mix."):
            return (H,), 0.0, 0.1  # norms
        shape = own[kinds[int(layer[1:])]][name[4:]]
        return shape, means.get(name[4:], 0.0), 0.3 if name.endswith("conv") else 0.02 if len(shape) == 2 else 0.1

    return StackModel(cfg, RandomTensors(torch, shape_of))


def zedotar_launches(torch, m, B, ctx):
    """Per-launch times of a step of B rows (B <= 16: single tokens at context ctx; else one prompt)."""
    from exo_amd import dense_ops as D
    from exo_amd.stack_config import MatrixMemorySpec

    c, prompt = m.cfg, B > 16
    H, eps = c.hidden_size, c.eps
    cache, bf, batch = launch_setup(torch, m, B, ctx)
    m._forward(cache, bf, batch, False)
    op = [bound[0] for bound in m._mixers(cache)]
    rows, fused = [], not prompt and D.post_linear_fits(B, m.layers[0].proj, bf.xb, H, True)
    other = torch.empty_like(bf.h)
    due = D.Branches(bf.branch, None)
    head = "residual, norm, " if fused else ""

    def add(name, fn, nbytes, flops, which=m.layers):
        fns = [(lambda L=L: fn(L)) for L in which]
        rows.append(row_of(name, time_launches(torch, fns * -(-12 // len(fns))), nbytes, flops))

    def mm(n, k):
        return 2 * n * k + 2 * B * (n + k), 2 * B * n * k

    def product(L, w, out, pre, **kw):
        if fused:
            D.post_linear(bf.h, due, eps, other, None, w, out, B, pre=pre, **kw)
        elif "up" in kw:
            D.glu(bf.xb, w, kw["up"], out, B, kw["spec"])
        else:
            D.linear(bf.xb, w, out, B, **kw)
    kind = {L.index: "memory" if isinstance(L.spec.mixer, MatrixMemorySpec) else "sigmoid" if L.spec.mixer.sigmoid else "window" for L in m.layers}
    for name in ("window", "sigmoid", "memory"):
        which = [L for L in m.layers if kind[L.index] == name]
        L0, s = which[0], which[0].spec.mixer
        p = L0.parts[0]
        y, y2 = bf.cols("proj", -(-L0.n_main // 8) * 8), bf.f32("proj_tail", -(-L0.n_tail // 8) * 8) if L0.n_tail else None
        add(f"{head}{name}: projection", lambda L: product(L, L.proj, y, L.pre1, bias=L.proj_b, tail=(y2, L.n_tail) if L.n_tail else None),
            *mm(L0.proj.shape[0], H), which)
        if name == "memory":
            h, _, d, _ = s.core
            e = s.vdim
            # at least: inputs and outputs once, the state in and out; two products with it per token
            add("memory: recurrence", lambda L: L.parts[0]._recur(op[L.index], bf, batch, h, True),
                B * (2 * h * (2 * d + e) + 4 * h * e) + 8 * h * d * (e + 1) * (1 if prompt else B), 4 * B * h * d * (e + 1), which)
            ro, oo, pk = bf.f32("recur", h * s.values), bf.mixed("recur_out", h * e), bf.f32("peaks", h)
            add("memory: divisor, gated norm", lambda L: D.gated_norm(ro, y[:, p.gate_col :], L.parts[0].norm, oo, B, h * e, h, eps, False,
                                                                    sigmoid=True, part=s.values, peaks=pk), B * h * e * 8, 0, which)
            src = oo
        else:
            seen = [i + 1 for i in range(B)] if prompt else [ctx] * B
            vis = [min(n, s.window) + max(0, n - s.window) // s.pool if s.window else n for n in seen]
            nk = 1 if s.shared_kv else 2  # columns of keys (and values) that come in
            kvb = 2 * s.kv_heads * (s.dim + s.vdim) * (B if prompt else sum(vis))
            fl = 2 * sum(vis) * s.heads * (s.dim + s.vdim)
            out = src = bf.mixed("attn", p.width)
            kw = dict(gate=y2[:, p.tcol :]) if s.head_gate else dict(out_gate=y[:, p.gate_col :])
            gb = 2 * B * p.width if s.out_gate else 0
            if prompt:
                q_out = bf.cols("queries", s.heads * s.dim) if s.conv else None
                q = y if q_out is None else q_out
                add(f"{name}: {'convolution, ' if s.conv else ''}turn; append{', means' if s.pool else ''}",
                    lambda L: op[L.index].append(y, batch.slot, batch.pos, B, q_out, *batch.means.get(s.pool, (None, 0))),
                    4 * B * s.heads * s.dim + kvb * (1 + nk / 2), 0, which)
                add(f"{name}: attention", lambda L: op[L.index].prompt(q, out, *batch.blocks[op[L0.index].prompt_block(s)], **kw),
                    kvb + 4 * B * s.heads * s.dim + gb, fl, which)
            else:
                add(f"{name}: {'convolution, ' if s.conv else ''}turn, append, attention",
                    lambda L: op[L.index].rows(y, out, batch.slot, batch.pos, B, batch.keys, append=True, **kw), kvb + gb, fl, which)
        add(f"{name}: o", lambda L: D.linear(src, L.parts[0].o, bf.branch, B), *mm(H, p.width), which)
    if not fused:
        add("residual + norm", lambda L: D.post_norm_add(due, eps, bf.h, bf.xb, B, L.pre2), B * H * 14, 0)
    f = c.layers[0].mlp
    act = bf.mixed("ff", f.ff)
    add(f"{head}gate, up", lambda L: product(L, L.ff.gate, act, L.pre2, up=L.ff.up, spec=f), *mm(2 * f.ff, H))
    add("down", lambda L: D.linear(act, L.ff.down, bf.branch, B), *mm(H, f.ff))
    return rows


def step_rates(torch, m, args, tag) -> dict:
    """Whole steps: prompt and decode throughput at batch 1, 4, 8 and 16."""
    from exo_amd.generate import prefill

    g = torch.Generator().manual_seed(1234)
    out = dict(weights_GB=round(m.weight_bytes() / 1e9, 2))
    prompt = torch.randint(0, m.cfg.vocab_size, (args.prompt,), generator=g).tolist()
    for B in (1, 4, 8, 16):
        cache = m.make_cache(B, args.prompt + args.steps + args.warmup + 64)
        for row in range(B):
            if row < 2:  # (the second time is the timed one: buffers and code objects are there)
                for _ in range(2):
                    cache.reset(rows=range(row, row + 1))
                    tps, n = prefill(m, prompt, cache, row=row, faithful_extra_steps=False)
                out["prefill_tok_s"], out["prefill_tokens"] = round(tps), n
            else:
                prefill(m, prompt, cache, row=row, faithful_extra_steps=False)
        bufs = m._buffers(B, 1)
        bufs.tokens.fill_(1)
        for _ in range(max(args.warmup, 1)):
            m.decode_step(cache, B, feedback=True)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(args.steps):
            m.decode_step(cache, B, feedback=True)
        torch.cuda.synchronize()
        dt = (time.perf_counter() - t0) / args.steps
        out[f"decode_tok_s_b{B}"], out[f"us_per_step_b{B}"] = round(B / dt, 1), round(dt * 1e6, 1)
        print(f"[bench] {tag} batch {B}: {dt * 1e6:.0f} us/step, prompt {out['prefill_tok_s']} tok/s", file=sys.stderr, flush=True)
        m._graphs.clear()
        del cache
    return out


def stack_workload(args):
    """A layer-list design beside the closest other model of equal size."""
    import torch

    from exo_amd import native

    native.load()
    torch.cuda.set_device(0)
    kinds = {"gekazen": (lambda size, name: gekazen_model(torch, size, 4096), gekazen_launches),
             "novosun": (lambda size, name: novosun_model(torch, size, NOVOSUN_SIZES[name]), novosun_launches),
             "pimisun": (lambda size, name: pimisun_model(torch, size, PIMISUN_SIZES[name]), pimisun_launches),
             "zedotar": (lambda size, name: zedotar_model(torch, size, NOVOSUN_SIZES[name], ZEDOTAR_SIZES[name]), zedotar_launches),
             "qwen3_moe": (lambda size, name: qwen_model(torch, size), qwen_launches)}
    pair = (args.workload, {"gekazen": "qwen3_moe", "zedotar": "novosun"}.get(args.workload, "gekazen"))
    report = {}
    for name in (GEKAZEN_SIZES if args.size == "all" else [args.size]):
        size, res = GEKAZEN_SIZES[name], {}
        for kind in pair:
            build, launches = kinds[kind]
            m = build(size, name)
            out = res[kind] = step_rates(torch, m, args, f"{name} {kind}")
            for B in (1, 8, args.prompt):
                out[f"launches_{B}_rows"] = launches(torch, m, B, args.prompt)
                for r in out[f"launches_{B}_rows"]:
                    print(f"[bench] {name} {kind} rows {B}: {r}", file=sys.stderr, flush=True)
            del m
            torch.cuda.empty_cache()
        report[name] = res
    first = next(iter(report.values()))[pair[0]]
    own = {"gekazen": {}, "novosun": NOVOSUN_SIZES, "pimisun": PIMISUN_SIZES, "zedotar": ZEDOTAR_SIZES}[args.workload]
    sizes = {k: GEKAZEN_SIZES[k] + own.get(k, ()) for k in report}
    print(json.dumps({
        "metric": f"decode tok/s, {pair[0].capitalize()} design, batch 1", "value": first["decode_tok_s_b1"], "unit": "tok/s",
        "n_gpus": 1, "steps": args.steps, "warmup": args.warmup, "ms_per_step": first["us_per_step_b1"] * 1e-3,
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "bf16", "data": "synthetic",
        "config": {"workload": f"{pair[0].capitalize()} layers of real size, random weights, context {args.prompt}, beside a "
                               f"{pair[1]} of equal size; x = launch time over its roofline", "sizes": sizes},
        "results": report}))


def main():
    args = parse_args()
    if args.gpus != 1:
        print(f"bench.py: this build runs on ONE GPU (per-shard forward); --gpus {args.gpus} is not "
              "supported: every figure here is one GPU's throughput.",
              file=sys.stderr)
        sys.exit(2)
    if args.workload == "qmatmul_sweep":
        return qmatmul_sweep(args)
    if args.workload in ("gekazen", "novosun", "pimisun", "zedotar"):
        return stack_workload(args)
    import torch

    from exo_amd import native
    from exo_amd.config import named_config
    from exo_amd.generate import prefill
    from exo_amd.model import ShardModel
    from exo_amd.synth import synth_weights

    native.load()  # fail loudly if the HIP library is missing
    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    cfg = named_config(args.config)
    if args.layers:
        cfg.num_hidden_layers = args.layers
    B = args.batch
    if not 1 <= B <= 16:
        sys.exit("bench.py: --batch must be 1..16")
    end = args.shard_layers or cfg.num_hidden_layers
    t0 = time.perf_counter()
    weights = synth_weights(cfg, 0, end, seed=0, device=dev)
    model = ShardModel(cfg, weights, 0, end, device=dev)
    del weights
    torch.cuda.synchronize()
    t_build = time.perf_counter() - t0
    print(f"[bench] weights ready in {t_build:.1f} s", file=sys.stderr, flush=True)

    g = torch.Generator().manual_seed(1234)
    K, W = args.steps, args.warmup
    cache = model.make_cache(B, args.prompt + K + W + 64)

    # prefill with the reference's protocol (one sequence at a time, as its batch engine
    # does), then the last-but-one prompt token of every sequence as a GEMV step
    tps_prefill, n_prefill, last = 0.0, 0, []
    for row in range(B):
        prompt = torch.randint(0, cfg.vocab_size, (args.prompt,), generator=g).tolist()
        # untimed warm-up of the same call (buffers, code objects, the captured single-token
        # step of this cache row, as in an engine whose cache outlives its requests), then rewind
        prefill(model, prompt[:-1], cache, row=row, faithful_extra_steps=model.is_last, graph_steps=True)
        cache.reset(rows=range(row, row + 1))
        tps, n = prefill(model, prompt[:-1], cache, row=row,
                         faithful_extra_steps=model.is_last, graph_steps=True)
        tps_prefill, n_prefill = tps, n
        model(torch.tensor([[prompt[-2]]], dtype=torch.int32), cache, logits="none",
              rows=slice(row, row + 1))
        last.append(prompt[-1])
        print(f"[bench] row {row}: prefill {n} tokens at {tps:.0f} tok/s", file=sys.stderr, flush=True)
    bufs = model._buffers(B, 1)
    bufs.tokens.copy_(torch.tensor(last, dtype=torch.int32))

    def step():
        return model.decode_step(cache, B, use_graph=not args.no_graph, feedback=model.is_last)

    for _ in range(W):
        step()
    torch.cuda.synchronize()
    ctx0 = cache[0].offset
    t0 = time.perf_counter()
    for _ in range(K):
        step()
    torch.cuda.synchronize()
    dt = time.perf_counter() - t0
    last_token = int(bufs.next_token[0]) if model.is_last else None
    tok_s = B * K / dt
    token_bytes = active_token_bytes(model, cfg, ctx0, B)

    if args.pmc_copy:
        # plain 16-byte-per-lane copy of 256 MiB (the KV re-layout kernel with one head is
        # exactly that): reads 256 MiB, writes 256 MiB
        from exo_amd import ops
        a = torch.zeros(1, 1 << 20, 128, dtype=torch.bfloat16, device=dev)
        ops.kv_export_nhd(a, 0, 1 << 20)
        torch.cuda.synchronize()
        del a

    headline = (args.config == "llama-3.1-8b" and B == 1 and model.is_last and not cfg.is_moe)
    if not cfg.is_moe and model.is_last and B == 1:
        # (a counter pass serialises every dispatch: one replay per region is plenty there)
        kernels = measure_kernels(model, torch, reps=1 if args.pmc_copy else 20)
        for k in kernels:
            k["frac_of_8TBps"] = k["GBps"] / 8000.0
            k["us_per_token"] = k["avg_us"] * k["launches_per_token"]
        dom = max(kernels, key=lambda k: k["us_per_token"])
        traffic, traffic_src = pmc_traffic(dom["name"]) if headline else (None, None)
        gemv_us = sum(k["us_per_token"] for k in kernels)
        gemv_bytes = sum(k["bytes_per_launch"] * k["launches_per_token"] for k in kernels)
        roofline = dict(bound="hbm", achieved=dom["GBps"], peak=8000.0, unit="GB/s",
                        frac=dom["GBps"] / 8000.0,
                        traffic=traffic, traffic_source=traffic_src, kernel=dom["kernel"],
                        launch=dom["name"], avg_us=dom["avg_us"], bytes_per_launch=dom["bytes_per_launch"],
                        all_gemv_GBps=gemv_bytes / gemv_us * 1e-3, all_gemv_us_per_token=gemv_us)
    else:
        # no single dominant launch is isolated here: the whole step against its bytes
        kernels = None
        gbps = token_bytes / (dt / K) * 1e-9
        roofline = dict(bound="hbm", achieved=gbps, peak=8000.0, unit="GB/s", frac=gbps / 8000.0,
                        traffic=None, kernel="all launches of one decode step",
                        bytes_per_launch=token_bytes, avg_us=dt / K * 1e6)

    engine = None
    if model.is_last and not args.no_engine:
        engine = engine_rates(model, cfg, args, torch)

    what = {"llama-3.2-1b": "configs[0]", "llama-3.1-8b": "configs[2]", "qwen3-30b-a3b": "configs[3]",
            "qwen3-235b-a22b": "configs[4]"}.get(args.config, "custom")
    shard = "" if model.is_last else f", pipeline shard of layers [0,{end}) (output: hidden state)"
    out = {
        "metric": ("decode tok/s + qmatmul HBM GB/s (% peak), Llama-3.1-8B 4-bit g64 bs1" if headline
                   else f"decode tok/s, {args.config} {cfg.bits}-bit g64 batch {B}"),
        "value": tok_s, "unit": "tok/s", "n_gpus": 1, "steps": K, "warmup": W,
        "ms_per_step": dt / K * 1e3, "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": "bf16", "data": "synthetic",
        "config": {"workload": f"{what}: {args.config} architecture, MLX affine {cfg.bits}-bit g64, "
                               f"random prompt of {args.prompt} tokens, greedy decode, batch {B}{shard}",
                   "layers": len(model.layers), "context_at_start": ctx0, "hip_graph": not args.no_graph},
        "roofline": roofline,
        "prefill_tok_s": tps_prefill, "prefill_tokens": n_prefill,
        "token_bytes": token_bytes, "effective_GBps": token_bytes * (K / dt) * 1e-9,
        "kernels": kernels, "build_s": t_build, "last_token": last_token,
    }
    if engine is not None:
        out.update(engine)
    if not args.no_cpu_baseline and kernels is not None:
        out["cpu_baseline"] = cpu_baseline(model, torch, args.cpu_seconds, ctx0)
    else:
        out["cpu_baseline"] = None
    print(json.dumps(out))


if __name__ == "__main__":
    main()
