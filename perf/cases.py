"""The work this framework is used for, as cases that can be timed through its public entry points.

Five kinds of call, each as a user's program makes it:

* ``linear``   -- one packed-weight product on device buffers (`kernels.DeviceWeight.matmul`): a decode step's products have
  one row, a batch of sequences or a speculative draft a few, a prompt tens to thousands;
* ``host``     -- the same product through the kernel SPI's calling convention: host arrays in and out, the weight resident
  (`kernels.HipRowMajorMatmulKernel.run`);
* ``attend``   -- fused attention over a KV cache (`kernels.sdpa_cache_dev`): one query per sequence in decode, a chunk of
  queries for a draft, a prompt in prefill;
* ``mlp``      -- one request against a dense fp32 network through the resident ops class (`ops.HipOps`): array up, layers,
  array down;
* ``decoder``  -- a Llama-shaped model (`decoder.LlamaDecoder`): prefill of a prompt, then decode steps over a given
  continuation (the tokens are given, not sampled, so that two implementations that round differently stay on one text).
"""
import numpy as np
import torch

from skainet_amd import kernels
from skainet_amd.decoder import DeviceBuffer, LayerWeights, LlamaConfig, LlamaDecoder, LlamaWeights
from skainet_amd.ops import ForwardScope, HipOps

SIGMA = 0.02      # weights are about N(0, 0.02^2), activations N(0, 1)


def listed():
    return [
        # the smallest product of the kernel benchmarks: all latency
        {"name": "q4k 1x1024x1024", "kind": "linear", "enc": "Q4_K", "m": 1, "n": 1024, "k": 1024},
        # the decode product the headline is quoted on: a 7B FFN projection, one token
        {"name": "q4k 1x11008x4096", "kind": "linear", "enc": "Q4_K", "m": 1, "n": 11008, "k": 4096},
        # the output head of a decode step
        {"name": "q6k 1x32000x4096", "kind": "linear", "enc": "Q6_K", "m": 1, "n": 32000, "k": 4096},
        # four sequences decoded together, down projection (rows of 11008: no power of two)
        {"name": "q8_0 4x4096x11008", "kind": "linear", "enc": "Q8_0", "m": 4, "n": 4096, "k": 11008},
        # a short chat prompt: more rows than the decode kernels take, fewer than a tile
        {"name": "q4k 24x14336x4096", "kind": "linear", "enc": "Q4_K", "m": 24, "n": 14336, "k": 4096},
        # the prompt product the headline is quoted on
        {"name": "q4k 512x4096x4096", "kind": "linear", "enc": "Q4_K", "m": 512, "n": 4096, "k": 4096},
        # a long prompt that is no multiple of any tile, in the second K-quant
        {"name": "q6k 1000x11008x4096", "kind": "linear", "enc": "Q6_K", "m": 1000, "n": 11008, "k": 4096},
        # a model that keeps its activations in host arrays and calls the SPI per linear layer
        {"name": "host q4k 1x4096x4096", "kind": "host", "enc": "Q4_K", "m": 1, "n": 4096, "k": 4096},
        # prompt attention, causal, grouped query heads
        {"name": "attend prompt 2048", "kind": "attend", "batch": 1, "heads": 32, "kv_heads": 8, "sq": 2048, "skv": 2048, "dim": 128,
         "window": 0},
        # decode attention of eight sequences over full caches
        {"name": "attend decode 8x4096", "kind": "attend", "batch": 8, "heads": 32, "kv_heads": 8, "sq": 1, "skv": 4096, "dim": 128,
         "window": 0},
        # a batch of requests against a dense three-layer network
        {"name": "mlp 32x1024-4096-1000", "kind": "mlp", "m": 32, "inputs": 1024, "hidden": 4096, "outputs": 1000},
        # a chat turn on the Llama-3-8B shape: a ragged prompt and the answer's first tokens
        {"name": "llama 8b 300+32", "kind": "decoder", "layers": 32, "hidden": 4096, "heads": 32, "kv_heads": 8, "dim": 128,
         "ffn": 14336, "vocab": 128256, "ctx": 2048, "prompt": 300, "steps": 32},
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return max(lo, min(hi, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    kind = rng.choice(["linear"] * 6 + ["host"] + ["attend"] * 3 + ["mlp"] + ["decoder"])
    if kind in ("linear", "host"):
        enc = rng.choice(["Q4_K"] * 4 + ["Q6_K"] * 2 + ["Q8_0"] * 2 + ["Q5_K", "Q4_0", "Q5_0", "Q5_1"])
        one = rng.random() < (0.3 if kind == "linear" else 0.7)
        m = 1 if one else _log(rng, 2, 1024 if kind == "linear" else 64)
        return {"kind": kind, "enc": enc, "m": m, "n": _log(rng, 512, 32000), "k": 256 * _log(rng, 2, 56)}
    if kind == "attend":
        dim = rng.choice([64, 128, 128])
        kv_heads = rng.choice([1, 2, 4, 8])
        heads = kv_heads * rng.choice([1, 2, 4, 8])
        form = rng.choice(["decode", "decode", "draft", "prompt", "prompt"])
        if form == "decode":
            batch, sq = _log(rng, 1, 16), 1
            skv = _log(rng, 64, 8192)
        elif form == "draft":
            batch, sq = _log(rng, 1, 4), rng.randint(2, 8)
            skv = sq + _log(rng, 64, 4096)
        else:
            batch, sq = 1, _log(rng, 16, 3000)
            skv = sq + rng.choice([0, 0, _log(rng, 64, 2048)])      # with the second form, a later chunk of a long prompt
        window = _log(rng, 128, 1024) if rng.random() < 0.2 else 0
        return {"kind": "attend", "batch": batch, "heads": heads, "kv_heads": kv_heads, "sq": sq, "skv": skv, "dim": dim,
                "window": window}
    if kind == "mlp":
        return {"kind": "mlp", "m": _log(rng, 1, 256), "inputs": _log(rng, 16, 4096), "hidden": _log(rng, 64, 8192),
                "outputs": _log(rng, 10, 2000)}
    dim = rng.choice([64, 128])
    hidden = 256 * _log(rng, 2, 14)
    heads = hidden // dim
    kv_heads = rng.choice([h for h in (1, 2, 4, 8) if heads % h == 0])
    return {"kind": "decoder", "layers": _log(rng, 2, 24), "hidden": hidden, "heads": heads, "kv_heads": kv_heads, "dim": dim,
            "ffn": 256 * max(1, round(hidden * rng.choice([2.67, 3.5]) / 256)), "vocab": _log(rng, 1000, 64000), "ctx": 1024,
            "prompt": _log(rng, 2, 512), "steps": _log(rng, 4, 32)}


# ---------------------------------------------------------------------------------------------- inputs

def _f16(values):
    return values.to(torch.float16).reshape(-1, 1).view(torch.uint8).reshape(-1, 2)


def _codes(gen, blocks, count, bits):
    """[blocks, count] codes of `bits` bits as a quantised Gaussian has them: +- 2.6 sigma over the range."""
    top = (1 << bits) - 1
    c = torch.randn((blocks, count), generator=gen, device="cuda")
    return c.mul_(top / 5.2).add_(top / 2).round_().clamp_(0, top).to(torch.uint8)


def _packed(enc, n, k, gen):
    """[n, k] weights, about N(0, SIGMA^2), as GGUF blocks: uint8 device bytes."""
    bs, nb = kernels.ENCODINGS[enc][1:]
    count = n * (k // bs)
    out = torch.empty((count, nb), dtype=torch.uint8, device="cuda")
    step = max(1, (1 << 26) // bs)
    for at in range(0, count, step):
        b = min(count, at + step) - at
        o = out[at:at + b]
        jitter = 1 + 0.1 * torch.rand((b, 1), generator=gen, device="cuda")
        if enc == "Q8_0":
            c = torch.randn((b, bs), generator=gen, device="cuda").mul_(127 / 2.6).round_().clamp_(-127, 127)
            o[:, :2] = _f16(jitter * (2.6 * SIGMA / 127))
            o[:, 2:] = c.to(torch.int8).view(torch.uint8)
        elif enc == "Q4_0":
            c = _codes(gen, b, bs, 4)
            o[:, :2] = _f16(jitter * (5.2 * SIGMA / 15))
            o[:, 2:] = c[:, :16] | (c[:, 16:] << 4)
        elif enc in ("Q5_0", "Q5_1"):
            c = _codes(gen, b, bs, 5)
            d = jitter * (5.2 * SIGMA / 31)
            o[:, :2] = _f16(d)
            at_h = 2
            if enc == "Q5_1":
                o[:, 2:4] = _f16(-15.5 * d)
                at_h = 4
            bit = 1 << torch.arange(8, device="cuda", dtype=torch.int32)
            o[:, at_h:at_h + 4] = ((c >> 4).to(torch.int32).reshape(b, 4, 8) * bit).sum(-1).to(torch.uint8)
            o[:, at_h + 4:] = (c[:, :16] & 15) | ((c[:, 16:] & 15) << 4)
        elif enc in ("Q4_K", "Q5_K"):
            bits = 4 if enc == "Q4_K" else 5
            c = _codes(gen, b, bs, bits).reshape(b, 4, 2, 32)
            d = jitter * (5.2 * SIGMA / ((1 << bits) - 1) / 48)
            o[:, :2] = _f16(d)
            o[:, 2:4] = _f16(d * ((1 << bits) - 1) / 2)
            s = torch.randint(36, 61, (b, 8), generator=gen, device="cuda", dtype=torch.int32)      # 6-bit scales; minima alike
            low, high = s[:, :4], s[:, 4:]
            o[:, 4:8] = (low | (high >> 4 << 6)).to(torch.uint8)
            o[:, 8:12] = (low | (high >> 4 << 6)).to(torch.uint8)
            o[:, 12:16] = ((high & 15) | ((high & 15) << 4)).to(torch.uint8)
            if enc == "Q5_K":
                h = (c >> 4).reshape(b, 8, 32)
                o[:, 16:48] = sum(h[:, g] << g for g in range(8))
                c = c & 15
            o[:, -128:] = (c[:, :, 0] | (c[:, :, 1] << 4)).reshape(b, 128)
        else:      # Q6_K
            c = _codes(gen, b, bs, 6).reshape(b, 2, 4, 32)
            lo, hi = c & 15, c >> 4
            o[:, :128] = torch.cat([lo[:, :, 0] | (lo[:, :, 2] << 4), lo[:, :, 1] | (lo[:, :, 3] << 4)], -1).reshape(b, 128)
            o[:, 128:192] = (hi[:, :, 0] | (hi[:, :, 1] << 2) | (hi[:, :, 2] << 4) | (hi[:, :, 3] << 6)).reshape(b, 64)
            s = torch.randint(70, 128, (b, 16), generator=gen, device="cuda", dtype=torch.int32)
            o[:, 192:208] = s.to(torch.uint8)
            o[:, 208:] = _f16(jitter * (5.2 * SIGMA / 63 / 99))
    return out.reshape(-1)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda")


def _model(case, gen):
    """A model of the case's shape: one layer's values, every layer in memory of its own."""
    cfg = LlamaConfig(layers=case["layers"], hidden=case["hidden"], heads=case["heads"], kv_heads=case["kv_heads"],
                      head_dim=case["dim"], ffn=case["ffn"], vocab=case["vocab"], ctx_max=case["ctx"])

    def gain():
        g = (1 + 0.1 * _randn(gen, cfg.hidden)).cpu().numpy()
        return DeviceBuffer(g.nbytes).upload(g)

    def weight(enc, rows, cols, values=None):
        values = _packed(enc, rows, cols, gen) if values is None else values.clone()
        return kernels.DeviceWeight.wrap(enc, values, rows, cols), values

    w = LlamaWeights.__new__(LlamaWeights)
    w.cfg, w.host, w.layers = cfg, None, []
    enc = cfg.linear_encoding
    w.tok_embd = weight(enc, cfg.vocab, cfg.hidden)[0]
    shapes = [(cfg.q_dim + 2 * cfg.kv_dim, cfg.hidden), (cfg.hidden, cfg.q_dim), (2 * cfg.ffn, cfg.hidden), (cfg.hidden, cfg.ffn)]
    first = [weight(enc, r, c) for r, c in shapes]
    for i in range(cfg.layers):
        q, o, g, d = [f[0] if i == 0 else weight(enc, r, c, f[1])[0] for f, (r, c) in zip(first, shapes)]
        w.layers.append(LayerWeights(attn_norm=gain(), wqkv=q, wo=o, ffn_norm=gain(), w_gate_up=g, w_down=d))
    w.out_norm = gain()
    w.head = weight(cfg.head_encoding, cfg.vocab, cfg.hidden)[0]
    return w


def prepare(case, seed):
    gen, kind = _gen(seed), case["kind"]
    s = {"case": case}
    if kind in ("linear", "host"):
        m, n, k = case["m"], case["n"], case["k"]
        packed, x = _packed(case["enc"], n, k, gen), _randn(gen, m, k)
        if kind == "linear":
            s.update(w=kernels.DeviceWeight.wrap(case["enc"], packed, n, k), x=x, out=torch.empty((m, n), device="cuda"))
        else:
            s.update(kernel=kernels.HipRowMajorMatmulKernel(case["enc"]), bytes=packed.cpu().numpy(), x=x.cpu().numpy(),
                     out=np.empty((m, n), np.float32))
    elif kind == "attend":
        b, h, hkv, sq, skv, d = (case[c] for c in ("batch", "heads", "kv_heads", "sq", "skv", "dim"))
        s.update(q=_randn(gen, b, h, sq, d), k=_randn(gen, b, hkv, skv, d), v=_randn(gen, b, hkv, skv, d),
                 out=torch.empty((b, h, sq, d), device="cuda"))
    elif kind == "mlp":
        ops, scope = HipOps(), ForwardScope(4 * case["m"] * (case["inputs"] + 8 * case["hidden"] + 4 * case["outputs"]) + (1 << 16))
        sizes = [case["inputs"], case["hidden"], case["hidden"], case["outputs"]]
        s["layers"] = [(ops.to_resident((_randn(gen, o, i) * i ** -0.5).cpu().numpy()), ops.to_resident((0.1 * _randn(gen, o)).cpu().numpy()))
                       for i, o in zip(sizes, sizes[1:])]
        s["norm"] = [ops.to_resident((c + 0.1 * _randn(gen, case["hidden"])).cpu().numpy()) for c in (1.0, 0.0)]
        s.update(ops=HipOps(scope), scope=scope, x=_randn(gen, case["m"], case["inputs"]).cpu().numpy())
    else:
        tokens = torch.randint(0, case["vocab"], (case["prompt"] + case["steps"],), generator=gen, device="cuda", dtype=torch.int32)
        s.update(decoder=LlamaDecoder(_model(case, gen), max_prefill=case["prompt"]), prompt=tokens[:case["prompt"]].cpu().numpy(),
                 next=tokens[case["prompt"]:].contiguous(), zero=torch.zeros(1, dtype=torch.int32, device="cuda"))
    return s


# ---------------------------------------------------------------------------------------------- one pass

def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "linear":
        s["w"].matmul(s["x"], case["m"], s["out"])
        return s["out"]
    if kind == "host":
        s["kernel"].run(s["x"], s["bytes"], case["n"], s["out"])
        return s["out"]
    if kind == "attend":
        kernels.sdpa_cache_dev(s["q"], s["k"], s["v"], s["out"], case["batch"], case["heads"], case["kv_heads"], case["sq"],
                               case["skv"], case["skv"], case["dim"], case["dim"] ** -0.5, True, case["window"])
        return s["out"]
    if kind == "mlp":
        ops = s["ops"]
        s["scope"].reset()
        h = ops.to_resident(s["x"])
        for i, (w, b) in enumerate(s["layers"]):
            h = ops.add(ops.matmul_weight_transposed(h, w), b)
            if i < 2:
                h = ops.gelu(h, approximate=True)
            if i == 1:
                h = ops.layer_norm(h, *s["norm"], 1e-5)
        return ops.softmax(h).numpy()
    dec = s["decoder"]
    dec.prefill(s["prompt"])
    first = dec.last_logits()
    at = s["next"].data_ptr()
    for i in range(case["steps"]):
        kernels.i32_store_at_dev(dec.token, s["zero"], 0, at + 4 * i)
        dec.run_steps(1)
    return {"after_prompt": first, "after_continuation": dec.last_logits()}


# ---------------------------------------------------------------------------------------------- what a pass is

def _packed_bytes(enc, n, k):
    _, bs, nb = kernels.ENCODINGS[enc]
    return n * (k // bs) * nb


def _attended(sq, skv, window):
    """Query-key pairs that a causal mask, and a window of keys where there is one, leaves."""
    first = skv - sq
    return sum(min(first + i + 1, window) if window else first + i + 1 for i in range(sq))


def work(case):
    kind = case["kind"]
    if kind in ("linear", "host"):
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": _packed_bytes(case["enc"], n, k) + 4 * m * (n + k), "flops": 2 * m * n * k}
    if kind == "attend":
        b, h, hkv, sq, skv, d, win = (case[c] for c in ("batch", "heads", "kv_heads", "sq", "skv", "dim", "window"))
        keys = min(skv, win + sq - 1) if win else skv
        return {"bytes": 4 * b * d * (2 * h * sq + 2 * hkv * keys), "flops": 4 * b * h * d * _attended(sq, skv, win)}
    if kind == "mlp":
        m, i, h, o = case["m"], case["inputs"], case["hidden"], case["outputs"]
        weights = i * h + h * h + h * o
        return {"bytes": 4 * (weights + 4 * h + o + m * (i + o)), "flops": 2 * m * weights}
    hid, ffn, d, L = case["hidden"], case["ffn"], case["dim"], case["layers"]
    p, t = case["prompt"], case["steps"]
    kv = case["kv_heads"] * d
    per_layer = (2 * hid + 2 * kv) * hid + 3 * hid * ffn
    head, head_bytes = case["vocab"] * hid, _packed_bytes("Q6_K", case["vocab"], hid)
    once = L * _packed_bytes("Q4_K", per_layer // hid, hid) + head_bytes
    pairs = _attended(p, p, 0) + _attended(t, p + t, 0)
    cache = sum(8 * L * kv * (p + i + 1) for i in range(t)) + 8 * L * kv * p
    return {"bytes": (t + 1) * once + cache, "flops": 2 * L * per_layer * (p + t) + 2 * head * (t + 1) + 4 * L * hid * pairs}


def tolerance(case):
    kind = case["kind"]
    if kind in ("linear", "host"):
        # up to 8 rows the products are of fp32 class; above, both operands are rounded to bf16
        return {"rel": 3e-5} if case["m"] <= 8 else {"rel": 6e-3}
    if kind == "attend":
        # prompt shapes run on bf16 operands
        return {"rel": 2e-5} if case["sq"] < 16 else {"rel": 1e-2}
    if kind == "mlp":
        return {"rel": 2e-5}
    # a prompt's products round to bf16, layer after layer
    return {"rel": 2e-2} if case["prompt"] > 8 else {"rel": 1e-3}
