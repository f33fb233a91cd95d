"""What a user of this engine has it do, as cases that can be timed and compared.

Three kinds, all through the model classes that the engines drive:

  decode   a quantised shard (``ShardModel.decode_step``, the captured single-token step) over sequences that
           already hold a context: eight steps, then the sequences go back to where they were
  prompt   a quantised shard's forward over a portion of a prompt (``ShardModel.__call__``), on an empty cache
           or behind a context
  requests a layer-list decoder (``StackModel``): ragged prompts admitted in one step, then captured single-token
           steps of all of them

Sizes are those of the architectures that the engine's configurations name, cut to a few layers: a pass then costs what a
pipeline shard of that many layers costs, and inputs are made in a second.  Weights are normal and quantised in groups of 64, the
context's keys and values are normal, ids are uniform.
"""

from __future__ import annotations

import math
from dataclasses import replace

import torch

from exo_amd.config import named_config
from exo_amd.model import ShardModel
from exo_amd.sampling import DeviceSampler, SamplerSettings
from exo_amd.stack_config import StackConfig, novosun_dict
from exo_amd.stack_model import StackModel

DEV = "cuda:0"
STEPS = 8     # decoded tokens of a pass
GROUP = 64    # elements that share a scale and a bias
BACK = 0.006  # of the weights that lead back into the residual: a layer changes it by a part of what it holds, as in trained models
FAMILIES = {"llama-1b": "llama-3.2-1b", "llama-8b": "llama-3.1-8b", "qwen-30b": "qwen3-30b-a3b", "qwen-235b": "qwen3-235b-a22b"}

# Novosun sizes: width, heads, kv heads, head size, linear attention heads / key size / value size, recurrence heads / value size /
# state / groups, feed-forward, vocabulary
STACKS = {
    1024: (16, 8, 64, 4, 128, 256, 32, 64, 128, 1, 2560, 65536),
    2048: (32, 4, 128, 4, 256, 512, 64, 64, 128, 1, 6912, 151936),
    4096: (64, 4, 128, 8, 256, 512, 128, 64, 128, 8, 13824, 151936),
}


def _decode(family, layers, rows, context, bits=4, part="whole", sampler="greedy"):
    return dict(kind="decode", family=family, bits=bits, layers=layers, part=part, rows=rows, context=context, sampler=sampler)


def _prompt(family, layers, tokens, past=0, bits=4, part="whole", rows=1):
    return dict(kind="prompt", family=family, bits=bits, layers=layers, part=part, rows=rows, tokens=tokens, past=past)


def _requests(width, layers, rows, tokens, steps, dtype="bf16"):
    return dict(kind="requests", width=width, layers=layers, rows=rows, tokens=tokens, steps=steps, dtype=dtype)


def listed():
    return [
        # a small assistant's answer to a short question: every launch is small
        dict(_decode("llama-1b", 16, 1, 128), name="decode 1b 1 row"),
        # one user's chat with the 8B model, sampled as requests are by default
        dict(_decode("llama-8b", 8, 1, 2048, sampler="draw"), name="decode 8b 1 row"),
        # the same model serving eight requests
        dict(_decode("llama-8b", 8, 8, 2050), name="decode 8b 8 rows"),
        # a full batch of long documents on a shard in the middle of a pipeline
        dict(_decode("llama-8b", 4, 16, 12289, part="middle"), name="decode 8b 16 long rows"),
        # a mixture of experts serving a few requests
        dict(_decode("qwen-30b", 6, 4, 1024, sampler="draw"), name="decode 30b 4 rows"),
        # one request on a pipeline shard of the large mixture of experts, 8-bit weights
        dict(_decode("qwen-235b", 3, 1, 4096, bits=8, part="middle"), name="decode 235b 8-bit 1 row"),
        # the usual prompt with its documents
        dict(_prompt("llama-8b", 4, 2047), name="prompt 8b 2047"),
        # a chat message of a few sentences
        dict(_prompt("llama-8b", 8, 61), name="prompt 8b 61"),
        # a prompt to the mixture of experts
        dict(_prompt("qwen-30b", 4, 1023), name="prompt 30b 1023"),
        # a late portion of a long document, 8-bit weights, on a shard in the middle of a pipeline
        dict(_prompt("llama-8b", 2, 4096, past=12288, bits=8, part="middle"), name="prompt 8b 8-bit 4096 late"),
        # a batch of requests to a layer-list decoder, from prompts to a few tokens
        dict(_requests(2048, 6, 4, 700, 8), name="requests 2k 4 rows"),
        # short requests to a small one in 32-bit mode
        dict(_requests(1024, 6, 2, 40, 16, "f32"), name="requests 1k f32 2 rows"),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    most = [work(c) for c in listed()]
    flops, nbytes = max(w["flops"] for w in most), max(w["bytes"] for w in most)
    while True:
        family = rng.choice(sorted(FAMILIES))
        bits, part = rng.choice([4, 4, 8]), rng.choice(["whole", "middle"])
        layers = _log(rng, 1, {"qwen-235b": 3, "qwen-30b": 6}.get(family, 8))
        pick = rng.random()
        if pick < 0.4:
            c = _decode(family, layers, _log(rng, 1, 16), _log(rng, 1, 16384), bits, part, rng.choice(["greedy", "draw"]))
        elif pick < 0.8:
            past = 0 if rng.random() < 0.5 else _log(rng, 1, 12288)
            c = _prompt(family, min(layers, 4), _log(rng, 9, 4096), past, bits, part, rng.choice([1, 1, 1, 2]))
        else:
            c = _requests(rng.choice(sorted(STACKS)), 2 * _log(rng, 1, 4), _log(rng, 1, 12), _log(rng, 1, 1200), rng.randint(1, 16),
                          rng.choice(["bf16", "bf16", "f32"]))
            if c["dtype"] == "f32":
                c["tokens"] = min(c["tokens"], 150)
        w = work(c)
        if w["flops"] <= flops and w["bytes"] <= nbytes and c.get("rows", 1) * c.get("context", 0) <= 16 * 12289:
            return c


# ------------------------------------------------------------------ sizes and work


def _config(c):
    """The architecture cut to the layers of the case, and the layers that the shard holds: all of them (with embedding and
    head), or those between a first and a last shard's."""
    cfg = named_config(FAMILIES[c["family"]])
    n = c["layers"]
    if c["part"] == "whole":
        return replace(cfg, num_hidden_layers=n, bits=c["bits"]), 0, n
    return replace(cfg, num_hidden_layers=n + 2, bits=c["bits"]), 1, 1 + n


def _lengths(c):
    """Ragged prompts: the longest, and shorter ones down to a single token."""
    return [max(1, c["tokens"] // (1, 3, 10, 1000)[r % 4] - 5 * (r // 4)) for r in range(c["rows"])]


def work(c):
    if c["kind"] == "requests":
        return _work_requests(c)
    cfg, _, _ = _config(c)
    H, Hq, Hkv, D, V, n = cfg.hidden_size, cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim, cfg.vocab_size, c["layers"]
    per = c["bits"] / 8 + 4 / GROUP  # bytes of a weight
    decode = c["kind"] == "decode"
    steps, rows, T = (STEPS, c["rows"], 1) if decode else (1, c["rows"], c["tokens"])
    past = c["context"] if decode else c["past"]
    R = rows * T                                                      # tokens of a step
    attn = H * D * (Hq + 2 * Hkv) + Hq * D * H
    if cfg.is_moe:
        one, E, k = 3 * H * cfg.moe_intermediate_size, cfg.num_experts, cfg.num_experts_per_tok
        read = attn + E * H + one * E * (1 - (1 - k / E) ** R)        # (experts that some token chooses, on average)
        used = attn + E * H + one * k
    else:
        read = used = attn + 3 * H * cfg.intermediate_size
    keys = past + (steps + 1) / 2 if decode else past + T             # that a step reads of each sequence
    pairs = rows * (keys if decode else T * past + T * (T + 1) / 2)   # of queries and keys
    nbytes = n * (read * per + 2 * rows * keys * Hkv * D * 2 + 2 * R * Hkv * D * 2)
    flops = n * (2 * used * R + 4 * Hq * D * pairs)
    if c["part"] == "whole":
        out = rows * V                                                # (a prompt's last logits)
        nbytes += H * V * per + 2 * out + R * H * per
        flops += 2 * rows * H * V
    else:
        nbytes += 2 * 2 * R * H
    return {"bytes": steps * nbytes, "flops": steps * flops}


def _work_requests(c):
    hq, hkv, hd, lh, ld, lv, sh, sv, sn, sg, ff, V = STACKS[c["width"]]
    W, size = c["width"], 2 if c["dtype"] == "bf16" else 4
    lens, rows, pairs = _lengths(c), c["rows"], c["layers"] // 2
    inner = sh * sv
    linear = W * lh * (2 * ld + 2 * lv) + lh * lv * W + 3 * W * ff
    both = W * hd * (hq + 2 * hkv) + hq * hd * W + W * (2 * inner + 2 * sg * sn + sh) + inner * W + 3 * W * ff
    weights = pairs * (linear + both)
    state = lh * ld * lv + sh * sn * sv                               # of a linear and a parallel layer, float32
    total = sum(lens) + rows * c["steps"]
    attn = sum((n + c["steps"]) * (n + c["steps"] + 1) / 2 for n in lens) * pairs * 4 * hq * hd
    kv = pairs * 2 * hkv * hd * size
    nbytes = (1 + c["steps"]) * ((weights + W * V) * size + rows * V * size)
    nbytes += c["steps"] * (rows * pairs * 2 * 4 * state + sum(lens) * kv) + sum(lens) * kv
    flops = 2 * weights * total + 2 * rows * W * V * (1 + c["steps"]) + attn + 4 * pairs * state * total
    return {"bytes": nbytes, "flops": flops}


def tolerance(c):
    # measured against the 64-bit results: 1.6e-6 and up to 7e-6 (drawn) in 32 bits; in bf16 0.004 to 0.023, growing with
    # the number of layers (each rounds what it adds, and the next ones carry that on)
    if c["kind"] == "requests":
        return {"rel": 8e-6, "max": 2e-4} if c["dtype"] == "f32" else {"rel": 0.03, "max": 0.6}
    return {"rel": 0.03, "max": 0.6}


# ------------------------------------------------------------------ inputs


def _quantise(gen, rows, K, bits, experts=0, std=0.02):
    """A random matrix in the checkpoint's layout: codes packed into 32-bit words, a scale and a bias per group."""
    top, per = 2**bits - 1, 32 // bits
    total = rows * max(1, experts)
    words = torch.empty(total, K // per, dtype=torch.int32, device=DEV)
    scales = torch.empty(total, K // GROUP, dtype=torch.bfloat16, device=DEV)
    biases = torch.empty_like(scales)
    slab = max(1, (1 << 27) // K)
    for r in range(0, total, slab):
        n = min(slab, total - r)
        w = torch.empty(n, K // GROUP, GROUP, device=DEV).normal_(0.0, std, generator=gen)
        lo, hi = w.amin(-1), w.amax(-1)
        s, b = ((hi - lo) / top).bfloat16(), lo.bfloat16()
        q = ((w - b.float()[..., None]) / s.float()[..., None]).round_().clamp_(0, top).to(torch.int32).view(n, K // per, per)
        packed = words[r : r + n].zero_()
        for i in range(per):
            packed |= q[..., i] << (bits * i)
        scales[r : r + n], biases[r : r + n] = s, b
    if experts:
        return tuple(t.view(experts, rows, -1) for t in (words, scales, biases))
    return words, scales, biases


def _shard_inputs(c, seed):
    """Weights by the checkpoint's names, and the inputs: ids or residual rows, the context's keys and values."""
    cfg, start, end = _config(c)
    g = torch.Generator(device=DEV).manual_seed(seed)
    H, Hq, Hkv, D, bits = cfg.hidden_size, cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim, cfg.bits
    w = {}

    def q(name, n, k, experts=0, std=0.02):
        w[name + ".weight"], w[name + ".scales"], w[name + ".biases"] = _quantise(g, n, k, bits, experts, std)

    def gain(name, n):
        w[name + ".weight"] = torch.empty(n, device=DEV).normal_(1.0, 0.1, generator=g).bfloat16()

    for i in range(start, end):
        p = f"model.layers.{i}."
        gain(p + "input_layernorm", H)
        gain(p + "post_attention_layernorm", H)
        q(p + "self_attn.q_proj", Hq * D, H)
        q(p + "self_attn.k_proj", Hkv * D, H)
        q(p + "self_attn.v_proj", Hkv * D, H)
        q(p + "self_attn.o_proj", H, Hq * D, std=BACK)
        if cfg.is_moe:
            gain(p + "self_attn.q_norm", D)
            gain(p + "self_attn.k_norm", D)
            E, ff = cfg.num_experts, cfg.moe_intermediate_size
            q(p + "mlp.gate", E, H)
            q(p + "mlp.switch_mlp.gate_proj", ff, H, E)
            q(p + "mlp.switch_mlp.up_proj", ff, H, E)
            q(p + "mlp.switch_mlp.down_proj", H, ff, E, std=BACK)
        else:
            q(p + "mlp.gate_proj", cfg.intermediate_size, H)
            q(p + "mlp.up_proj", cfg.intermediate_size, H)
            q(p + "mlp.down_proj", H, cfg.intermediate_size, std=BACK)
    whole = c["part"] == "whole"
    if whole:
        # (smaller vectors where they are the head too)
        q("model.embed_tokens", cfg.vocab_size, H, std=0.3 if cfg.tie_word_embeddings else 1.0)
        gain("model.norm", H)
        if not cfg.tie_word_embeddings:
            q("lm_head", cfg.vocab_size, H)
    rows, T = c["rows"], STEPS if c["kind"] == "decode" else c["tokens"]
    past = c["context"] if c["kind"] == "decode" else c["past"]
    if whole:
        x = torch.randint(0, cfg.vocab_size, (rows, T), generator=g, device=DEV, dtype=torch.int32)
    else:
        x = torch.empty(rows, T, H, device=DEV).normal_(generator=g).bfloat16()
    kv = [torch.empty(rows, 2, Hkv, past, D, device=DEV, dtype=torch.bfloat16).normal_(generator=g) for _ in range(start, end)]
    return cfg, start, end, w, x, kv


def prepare(c, seed):
    if c["kind"] == "requests":
        return _prepare_requests(c, seed)
    cfg, start, end, w, x, kv = _shard_inputs(c, seed)
    model = ShardModel(cfg, w, start, end, device=DEV)
    rows, past = c["rows"], kv[0].shape[3]
    T = x.shape[1]
    cache = model.make_cache(rows, past + T + 64)
    for r in range(rows):
        cache.restore(r, [layer[r] for layer in kv], past)
    s = dict(case=c, model=model, cache=cache, x=x, sampler=None, mode=0)
    if c["kind"] == "prompt":
        return s
    s["x"] = x.transpose(0, 1).contiguous()  # step by step
    if c["sampler"] == "draw" and c["part"] == "whole":
        s["sampler"] = DeviceSampler(rows, cfg.vocab_size, DEV)
        for r in range(rows):
            s["sampler"].set_row(r, SamplerSettings(temperature=0.7, top_p=0.95, min_p=0.05, seed=seed + r), [1, 2, 3])
        s["mode"] = s["sampler"].mode(rows, want_top=True)
    # the engine's warm-up step: it captures the step's graph and hands out the buffers that the step reads and writes
    s["bufs"] = model.decode_step(cache, rows, sampler=s["sampler"], mode=s["mode"])
    cache.trim(1)
    return s


def _stack_weights(c, seed):
    W = c["width"]
    hq, hkv, hd, lh, ld, lv, sh, sv, sn, sg, ff, V = STACKS[W]
    kinds = "gp" * (c["layers"] // 2)
    d = novosun_dict(W, V, kinds, heads=hq, kv_heads=hkv, dim=hd, vdim=hd, ff=ff, lin_heads=lh, lin_dim=ld, lin_vdim=lv, ssm_heads=sh,
                     ssm_vdim=sv, ssm_state=sn, ssm_groups=sg, mult=0.5)
    g = torch.Generator(device=DEV).manual_seed(seed)
    w = {}

    def put(name, *shape, std=0.02, mean=0.0):
        w[name] = torch.empty(*shape, device=DEV, dtype=torch.bfloat16).normal_(mean, std, generator=g)

    def gain(name, n):
        put(name, n, std=0.1, mean=1.0)

    inner = sh * sv
    ch = inner + 2 * sg * sn
    put("embed", V, W)
    put("head", V, W)
    gain("final.norm", W)
    for i, kind in enumerate(kinds):
        p = f"l{i}."
        for n in ("norm1", "norm1b", "norm2", "norm2b"):
            gain(p + n, W)
        if kind == "g":
            p += "mix."
            for n, rows in (("q", lh * ld), ("k", lh * ld), ("v", lh * lv), ("g", lh * lv), ("a1", 16)):
                put(p + n, rows, W)
            put(p + "o", W, lh * lv)
            gain(p + "norm", lv)
            put(p + "a2", lh * ld, 16, std=0.3)
            put(p + "a2.b", lh * ld, std=0.5, mean=2.0)
        else:
            q = p + "mix.left."
            for n, rows in (("q", hq * hd), ("k", hkv * hd), ("v", hkv * hd), ("g", hq)):
                put(q + n, rows, W)
            gain(q + "q.norm", hd)
            gain(q + "k.norm", hd)
            put(q + "o", W, hq * hd)
            gain(q + "out", W)
            q = p + "mix.right."
            put(q + "in", inner + ch + sh, W)
            put(q + "conv", ch, 4, std=0.3)
            put(q + "conv.b", ch, std=0.1)
            put(q + "dt_bias", sh, std=0.5, mean=-3.0)
            put(q + "A_log", sh, std=0.5)
            put(q + "D", sh, std=0.5, mean=1.0)
            gain(q + "norm", inner)
            put(q + "o", W, inner)
            gain(q + "out", W)
        p = f"l{i}.mlp."
        put(p + "gate", ff, W)
        put(p + "up", ff, W)
        put(p + "down", W, ff)
    lens = _lengths(c)
    prompts = [torch.randint(0, V, (n,), generator=g, device=DEV, dtype=torch.int32) for n in lens]
    answers = torch.randint(0, V, (c["steps"], c["rows"]), generator=g, device=DEV, dtype=torch.int32)
    return d, w, prompts, answers


def _prepare_requests(c, seed):
    d, w, prompts, answers = _stack_weights(c, seed)
    model = StackModel(StackConfig.from_dict(d), w, device=DEV, dtype=torch.bfloat16 if c["dtype"] == "bf16" else torch.float32)
    cache = model.make_cache(c["rows"], max(_lengths(c)) + c["steps"] + 64)
    lists = [(r, p.tolist(), [len(p) - 1]) for r, p in enumerate(prompts)]
    s = dict(case=c, model=model, cache=cache, prompts=lists, answers=answers, bufs=None)
    # the engine's warm-up: a step of prompts, and the captured step of single tokens
    model.step(cache, lists)
    s["bufs"] = model.decode_step(cache, c["rows"])
    cache.reset()
    return s


# ------------------------------------------------------------------ the pass


def run(s):
    c, model, cache = s["case"], s["model"], s["cache"]
    if c["kind"] == "prompt":
        whole = c["part"] == "whole"
        past = c["past"]
        out = model(s["x"] if whole else None, cache, input_embeddings=None if whole else s["x"], logits="last")
        keys = [cache[i].keys[:, :, past : past + c["tokens"]].clone() for i in (0, len(cache) - 1)]
        cache.trim(c["tokens"])
        return {"out": out, "keys": keys}
    rows, bufs, outs, lses = c["rows"], s["bufs"], [], []
    if c["kind"] == "requests":
        outs.append(model.step(cache, s["prompts"]).clone())
        for ids in s["answers"]:
            bufs.tokens.copy_(ids)
            model.decode_step(cache, rows)
            outs.append(bufs.logits.clone())
        cache.reset()
        return {"logits": torch.stack(outs)}
    whole, sampler = c["part"] == "whole", s["sampler"]
    for x in s["x"]:
        (bufs.tokens if whole else bufs.h).copy_(x)
        model.decode_step(cache, rows, sampler=sampler, mode=s["mode"])
        outs.append((bufs.logits if whole else bufs.h).clone())
        if whole:
            lses.append((bufs if sampler is None else sampler).lse.clone())
    cache.trim(STEPS)
    out = {"out": torch.stack(outs)}
    if whole:
        out["lse"] = torch.stack(lses)
    if sampler is not None:
        out["top"] = sampler.top_val.clone()
    return out


# ------------------------------------------------------------------ the same in 64 bits


def _dequantise(w, name, bits, expert=None):
    words, s, b = (w[f"{name}.{n}"] if expert is None else w[f"{name}.{n}"][expert] for n in ("weight", "scales", "biases"))
    per = 32 // bits
    q = (words[..., None] >> torch.arange(0, 32, bits, device=DEV, dtype=torch.int32)) & (2**bits - 1)
    q = q.view(*words.shape[:-1], words.shape[-1] * per // GROUP, GROUP).double()
    return (q * s.double()[..., None] + b.double()[..., None]).flatten(-2)


def _rms(x, gain, eps):
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt() * gain.double()


def _frequencies(cfg):
    inv = cfg.rope_theta ** (-torch.arange(0, cfg.head_dim, 2, dtype=torch.float64, device=DEV) / cfg.head_dim)
    sc = cfg.rope_scaling
    if sc:
        turns = sc["original_max_position_embeddings"] * inv / (2 * math.pi)  # inside the original context
        lo, hi = sc["low_freq_factor"], sc["high_freq_factor"]
        mix = ((turns - lo) / (hi - lo)).clamp(0, 1)
        inv = inv * (mix + (1 - mix) / sc["factor"])
    return inv


def _rotate(x, pos, inv):
    a = pos.double()[:, None] * inv
    cos, sin = a.cos()[:, None], a.sin()[:, None]
    lo, hi = x.chunk(2, -1)
    return torch.cat([lo * cos - hi * sin, hi * cos + lo * sin], -1)


def _causal(q, k, v, past, scale):
    """q [T, Hq, D], k and v [G, past + T, D] -> [T, Hq, D]."""
    T, Hq, _ = q.shape
    per, n = Hq // k.shape[0], k.shape[1]
    allowed = torch.arange(n, device=DEV) <= torch.arange(T, device=DEV)[:, None] + past
    out = torch.empty(T, Hq, v.shape[-1], dtype=torch.float64, device=DEV)
    for h in range(Hq):
        s = (q[:, h] @ k[h // per].T) * scale
        s.masked_fill_(~allowed, -math.inf)
        out[:, h] = s.softmax(-1) @ v[h // per]
    return out


def _experts(cfg, w, p, x):
    probs = (x @ _dequantise(w, p + "mlp.gate", cfg.bits).T).softmax(-1)
    val, idx = probs.topk(cfg.num_experts_per_tok, -1)
    if cfg.norm_topk_prob:
        val = val / val.sum(-1, keepdim=True)
    y = torch.zeros_like(x)
    for e in idx.unique().tolist():
        row, slot = (idx == e).nonzero(as_tuple=True)
        g, u, d = (_dequantise(w, p + f"mlp.switch_mlp.{n}_proj", cfg.bits, e) for n in ("gate", "up", "down"))
        t = x[row]
        y.index_add_(0, row, (torch.nn.functional.silu(t @ g.T) * (t @ u.T)) @ d.T * val[row, slot][:, None])
    return y


def exact(c, seed):
    if c["kind"] == "requests":
        return _exact_requests(c, seed)
    cfg, start, end, w, x, kv = _shard_inputs(c, seed)
    Hq, Hkv, D, eps, bits = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim, cfg.rms_norm_eps, cfg.bits
    rows, T = x.shape[:2]
    past, whole, inv = kv[0].shape[3], c["part"] == "whole", _frequencies(cfg)
    embed = _dequantise(w, "model.embed_tokens", bits) if whole else None
    h = (embed[x.long()] if whole else x.double()).view(rows * T, -1)
    pos = torch.arange(past, past + T, device=DEV)
    keys = []
    for i in range(start, end):
        p = f"model.layers.{i}."
        n = _rms(h, w[p + "input_layernorm.weight"], eps)
        q, k, v = ((n @ _dequantise(w, p + f"self_attn.{a}_proj", bits).T).view(rows, T, -1, D) for a in "qkv")
        if cfg.is_moe:
            q, k = (_rms(t, w[p + f"self_attn.{a}_norm.weight"], eps) for t, a in ((q, "q"), (k, "k")))
        out, new = [], []
        for r in range(rows):
            kr = _rotate(k[r], pos, inv).transpose(0, 1)
            new.append(kr)
            ks, vs = torch.cat([kv[i - start][r, 0].double(), kr], 1), torch.cat([kv[i - start][r, 1].double(), v[r].transpose(0, 1)], 1)
            out.append(_causal(_rotate(q[r], pos, inv), ks, vs, past, D**-0.5).flatten(1))
        if i in (start, end - 1):
            keys.append(torch.stack(new))
        h = h + torch.cat(out) @ _dequantise(w, p + "self_attn.o_proj", bits).T
        n = _rms(h, w[p + "post_attention_layernorm.weight"], eps)
        if cfg.is_moe:
            h = h + _experts(cfg, w, p, n)
        else:
            g, u, d = (_dequantise(w, p + f"mlp.{a}_proj", bits) for a in ("gate", "up", "down"))
            h = h + (torch.nn.functional.silu(n @ g.T) * (n @ u.T)) @ d.T
    h = h.view(rows, T, -1)
    if c["kind"] == "prompt" and whole:
        h = h[:, -1:]
    if whole:
        head = embed if cfg.tie_word_embeddings else _dequantise(w, "lm_head", bits)
        h = _rms(h, w["model.norm.weight"], eps) @ head.T
    if c["kind"] == "prompt":
        return {"out": h, "keys": keys if len(keys) > 1 else keys * 2}
    h = h.transpose(0, 1).contiguous()
    out = {"out": h}
    if whole:
        out["lse"] = h.logsumexp(-1)
        if c["sampler"] == "draw":
            out["top"] = h[-1].topk(20, -1)[0] - out["lse"][-1][:, None]
    return out


def _recurrence(q, k, v, decay):
    """S <- diag(decay) S + k v^T, o = S^T q per head; q, k, decay [T, H, D], v [T, H, E] -> [T, H, E]."""
    S = torch.zeros(k.shape[1], k.shape[2], v.shape[2], dtype=torch.float64, device=DEV)
    out = torch.empty_like(v)
    for t in range(len(q)):
        S = decay[t][..., None] * S + k[t][..., None] * v[t][:, None]
        out[t] = (q[t][:, None] @ S)[:, 0]
    return out


def _exact_requests(c, seed):
    F = torch.nn.functional
    d, w16, prompts, answers = _stack_weights(c, seed)
    hq, hkv, hd, lh, ld, lv, sh, sv, sn, sg, ff, V = STACKS[c["width"]]
    eps, mult, inner = d["norm"]["eps"], d["residual_mult"], sh * sv
    outs = []
    for r, prompt in enumerate(prompts):
        ids = torch.cat([prompt, answers[:, r]]).long()
        T, w = len(ids), {}
        x = w16["embed"][ids].double()
        for i, L in enumerate(d["layers"]):
            p = f"l{i}."
            w = {k[len(p) :]: t.double() for k, t in w16.items() if k.startswith(p)}
            h = _rms(x, w["norm1"], eps)
            if L["type"] == "gla":
                q, k, v = ((h @ w[f"mix.{n}"].T).view(T, lh, -1) for n in "qkv")
                z = (h @ w["mix.a1"].T) @ w["mix.a2"].T + w["mix.a2.b"]
                a = (F.logsigmoid(z) / L["mixer"]["tau"]).exp().view(T, lh, ld)
                o = _rms(_recurrence(q / ld**0.5, k, v, a), w["mix.norm"], eps).reshape(T, -1)
                o = (o * F.silu(h @ w["mix.g"].T)) @ w["mix.o"].T
            else:
                q, k, v = ((h @ w[f"mix.left.{n}"].T).view(T, -1, hd) for n in "qkv")
                q, k = _rms(q, w["mix.left.q.norm"], eps), _rms(k, w["mix.left.k.norm"], eps)
                o = _causal(q, k.transpose(0, 1), v.transpose(0, 1), 0, hd**-0.5)
                o = (o * (h @ w["mix.left.g"].T).sigmoid()[..., None]).reshape(T, -1)
                left = _rms(o @ w["mix.left.o"].T, w["mix.left.out"], eps)
                z, u, dt = (h @ w["mix.right.in"].T).split([inner, inner + 2 * sg * sn, sh], 1)
                taps = w["mix.right.conv"]
                u = F.pad(u, (0, 0, taps.shape[1] - 1, 0))
                u = sum(u[j : j + T] * taps[:, j] for j in range(taps.shape[1])) + w["mix.right.conv.b"]
                u = F.silu(u)
                v = u[:, :inner].view(T, sh, sv)
                k, q = (t.view(T, sg, sn).repeat_interleave(sh // sg, 1) for t in u[:, inner:].chunk(2, 1))
                dt = F.softplus(dt + w["mix.right.dt_bias"])
                a = (-w["mix.right.A_log"].exp() * dt).exp()[..., None].expand(T, sh, sn)
                o = _recurrence(q, k, dt[..., None] * v, a) + w["mix.right.D"][:, None] * v
                o = o.reshape(T, inner) * F.silu(z)
                right = _rms(_rms(o, w["mix.right.norm"], eps) @ w["mix.right.o"].T, w["mix.right.out"], eps)
                o = (left + right) / 2
            x = x + mult * _rms(o, w["norm1b"], eps)
            h = _rms(x, w["norm2"], eps)
            g, u = (h @ w["mlp.gate"].T).clamp(max=L["mlp"]["limit"]), (h @ w["mlp.up"].T).clamp(-L["mlp"]["limit"], L["mlp"]["limit"])
            o = (g * (1.702 * g).sigmoid() * (u + 1)) @ w["mlp.down"].T
            x = x + mult * _rms(o, w["norm2b"], eps)
        outs.append(_rms(x[len(prompt) - 1 :], w16["final.norm"], eps) @ w16["head"].double().T)
    return {"logits": torch.stack(outs, 1)}
