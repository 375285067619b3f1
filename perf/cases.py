"""What this framework is timed on: its W8 linears, its attentions and its two
model plans, each through the public entry point a program calls.

A case is a dict of plain values; ``prepare`` makes the inputs and the handles
a program would hold (weights, packed copies, compiled plans), ``run`` makes
one pass and returns its outputs whole, ``exact`` the same outputs from plain
torch in 64 bits, ``work`` the bytes and operations a pass cannot do without.
"""
import math

import torch

import rxla_amd as rx

DEV = "cuda"

# Widths [n, k] of the dense decoder (hidden 2048, intermediate 6144), of the
# 0.8B hybrid model (hidden 1024, intermediate 3584) and of the 4096-wide layers.
WIDTHS = [(2048, 2048), (4096, 2048), (12288, 2048), (2048, 6144), (1024, 1024), (7168, 1024),
          (1024, 2048), (1024, 3584), (4096, 4096), (6144, 4096), (12288, 4096), (24576, 4096),
          (4096, 12288)]
# The hybrid model's projections, the ones that run with F32 compute.
F32_WIDTHS = [(8192, 1024), (7168, 1024), (5120, 1024), (1024, 2048), (1024, 3584)]
# (query heads, kv heads) from one query head per kv head to eight.
HEADS = [(8, 8), (16, 8), (8, 2), (32, 8), (16, 2), (32, 4), (64, 8)]


def listed():
    return [
        # one token through the dense decoder's attention output projection:
        # the smallest call, latency counts
        dict(name="linear-step", kind="linear", rows=1, n=2048, k=2048, group=0, x="bf16",
             packed=True, compute="bf16"),
        # a batch of 16 sequences, one token each, through a wide gate|up projection
        dict(name="linear-batch", kind="linear", rows=16, n=24576, k=4096, group=0, x="bf16",
             packed=True, compute="bf16"),
        # 48 rows (a short prompt, or several tokens for each of a few sequences)
        # over the checkpoint's own layout: row-major codes, 128-wide groups, f32 input
        dict(name="linear-chunk", kind="linear", rows=48, n=6144, k=4096, group=128, x="f32",
             packed=False, compute="bf16"),
        # a prompt of 2048 tokens through an MLP projection
        dict(name="linear-prompt", kind="linear", rows=2048, n=12288, k=4096, group=0, x="bf16",
             packed=False, compute="bf16"),
        # the reference's default compute type: gate|up of the 0.8B model, 16 tokens
        dict(name="linear-f32", kind="linear", rows=16, n=7168, k=1024, group=128, x="f32",
             packed=True, compute="f32"),
        # logits of a batch of 8 from the tied bf16 embedding
        dict(name="head", kind="head", rows=8, n=151936, k=2048, packed=True),
        # a decode step over long bf16 caches of ragged lengths
        dict(name="decode-attention", kind="decode", batch=8, q_heads=32, kv_heads=8, dim=128,
             low=512, cap=8192, cache="bf16", q="bf16"),
        # the same step over f32 caches, the type the reference keeps them in, with the
        # head width of the hybrid model's attention layers
        dict(name="decode-attention-f32", kind="decode", batch=4, q_heads=8, kv_heads=2, dim=256,
             low=300, cap=2048, cache="f32", q="f32"),
        # prompts that continue earlier ones, an odd number of rows each
        dict(name="prefill-attention", kind="prefill", batch=4, rows=777, start=500, q_heads=32,
             kv_heads=8, dim=128, q="bf16"),
        # the reference's own attention operator: f32 operands and an additive mask
        dict(name="masked-attention", kind="masked", batch=1, q_heads=16, kv_heads=8, queries=512,
             keys=512, dim=128, mask="causal"),
        # the 0.8B hybrid model on one prompt, logits of every position
        dict(name="hybrid-model", kind="hybrid", batch=1, tokens=500),
        # four layers of the dense decoder: a batch of prompts, then single-token steps
        dict(name="dense-decoder", kind="decoder", batch=8, prompt=128, steps=8, layers=4),
    ]


def _log(rng, low, high):
    """A whole number between low and high, spread over its logarithm."""
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "linear-f32", "head", "decode", "decode",
                       "prefill", "masked", "masked", "hybrid", "decoder"])
    if kind == "linear":
        # rows from one token to a long prompt; now and then a width between the listed ones
        n, k = rng.choice(WIDTHS)
        if rng.random() < 0.25:
            n = 16 * _log(rng, 40, 1000)
        rows = min(_log(rng, 1, 2048), 2048 * 12288 * 4096 // (n * k))
        # packed copies serve the decode sizes; prompts come with either layout
        packed = n % 128 == 0 and rng.random() < 0.5
        return dict(kind="linear", rows=rows, n=n, k=k, group=rng.choice([0, 0, 128]),
                    x=rng.choice(["bf16", "f32"]), packed=packed, compute="bf16")
    if kind == "linear-f32":
        n, k = rng.choice(F32_WIDTHS)
        return dict(kind="linear", rows=_log(rng, 1, 1024), n=n, k=k, group=128, x="f32",
                    packed=rng.random() < 0.5, compute="f32")
    if kind == "head":
        return dict(kind="head", rows=_log(rng, 1, 64), n=16 * _log(rng, 1000, 9496),
                    k=rng.choice([1024, 2048]), packed=rng.random() < 0.5)
    if kind == "decode":
        hq, hkv = rng.choice(HEADS)
        dim = rng.choice([64, 128, 128, 256])
        cap = _log(rng, 64, 8192)
        cache = rng.choice(["bf16", "bf16", "f32"])
        # at most the listed long caches' bytes
        per = hkv * dim * (2 if cache == "bf16" else 4)
        most = max(1, min(16, 8 * 8192 * 8 * 128 * 2 // (cap * per)))
        return dict(kind="decode", batch=rng.randint(1, most), q_heads=hq, kv_heads=hkv, dim=dim,
                    low=max(1, cap // rng.choice([2, 4, 16])), cap=cap, cache=cache,
                    q=rng.choice(["bf16", "f32"]))
    if kind == "prefill":
        hq, hkv = rng.choice(HEADS)
        dim = rng.choice([64, 128, 128, 256])
        rows = _log(rng, 16, 1024)
        start = rng.choice([0, 0, _log(rng, 1, 1024)])
        most = max(1, min(8, 4 * 777 * 32 * 128 * 1277 // (rows * hq * dim * (rows + start))))
        return dict(kind="prefill", batch=rng.randint(1, most), rows=rows, start=start, q_heads=hq,
                    kv_heads=hkv, dim=dim, q=rng.choice(["bf16", "f32"]))
    if kind == "masked":
        hq, hkv = rng.choice(HEADS[:4])
        dim = rng.choice([64, 128, 256])
        mask = rng.choice(["causal", "padding", "none"])
        keys = _log(rng, 16, 1024)
        queries = rng.choice([1, keys, min(keys, _log(rng, 2, 512))])
        most = max(1, min(8, 2 ** 33 // (queries * keys * hq * dim)))
        return dict(kind="masked", batch=rng.randint(1, most), q_heads=hq, kv_heads=hkv,
                    queries=queries, keys=keys, dim=dim, mask=mask)
    if kind == "hybrid":
        batch = rng.choice([1, 1, 2])
        return dict(kind="hybrid", batch=batch, tokens=_log(rng, 1, 500 // batch))
    return dict(kind="decoder", batch=rng.randint(1, 8), prompt=_log(rng, 1, 128),
                steps=rng.randint(1, 8), layers=4)


# ---- inputs ---------------------------------------------------------------------

_rt = None


def _runtime():
    global _rt
    if _rt is None:
        _rt = rx.Runtime(0)
    return _rt


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=DEV) * std


_FLOAT = {"bf16": torch.bfloat16, "f32": torch.float32}


def _codes(g, n, k, group, std=0.02):
    """A weight ~ N(0, std) as the encoder stores it: U8 codes (int8 + 128) and
    f32 scales, one per row or per group of the row."""
    width = group or k
    w = _normal(g, n, k // width, width, std=std)
    s = w.abs().amax(dim=2).clamp_min(1e-12) / 127
    q = (w / s[:, :, None]).round().clamp(-127, 127) + 128
    return q.to(torch.uint8).reshape(n, k), s.contiguous()


def _weights(u8, s, dtype=torch.float64):
    n, k = u8.shape
    w = (u8.to(dtype) - 128).reshape(n, s.shape[1], -1) * s.to(dtype)[:, :, None]
    return w.reshape(n, k)


def _linear_inputs(case, seed):
    g = _gen(seed)
    x = _normal(g, case["rows"], case["k"]).to(_FLOAT[case["x"]])
    u8, s = _codes(g, case["n"], case["k"], case["group"])
    return x, u8, s


def _head_inputs(case, seed):
    g = _gen(seed)
    x = _normal(g, case["rows"], case["k"]).bfloat16()
    return x, _normal(g, case["n"], case["k"], std=0.02).bfloat16()


def _decode_inputs(case, seed):
    g = _gen(seed)
    b, hq, hkv, d, cap = (case[k] for k in ("batch", "q_heads", "kv_heads", "dim", "cap"))
    q = _normal(g, b, hq, d).to(_FLOAT[case["q"]])
    kc = _normal(g, b, hkv, cap, d).to(_FLOAT[case["cache"]])
    vc = _normal(g, b, hkv, cap, d).to(_FLOAT[case["cache"]])
    lens = torch.randint(case["low"], cap + 1, (b,), generator=g, device=DEV, dtype=torch.int32)
    return q, kc, vc, lens


def _prefill_inputs(case, seed):
    g = _gen(seed)
    b, s, hq, hkv, d = (case[k] for k in ("batch", "rows", "q_heads", "kv_heads", "dim"))
    cap = case["start"] + s
    q = _normal(g, b, s, hq, d).to(_FLOAT[case["q"]])
    kc = _normal(g, b, hkv, cap, d).bfloat16()
    vc = _normal(g, b, hkv, cap, d).bfloat16()
    starts = torch.randint(case["start"] // 2, case["start"] + 1, (b,), generator=g, device=DEV,
                           dtype=torch.int32)
    return q, kc, vc, starts


def _masked_inputs(case, seed):
    g = _gen(seed)
    b, hq, hkv, sq, sk, d = (case[k] for k in ("batch", "q_heads", "kv_heads", "queries", "keys",
                                               "dim"))
    q, k, v = _normal(g, b, hq, sq, d), _normal(g, b, hkv, sk, d), _normal(g, b, hkv, sk, d)
    mask = None
    if case["mask"] == "causal":  # the last sq positions of sk
        mask = torch.zeros(sq, sk, device=DEV).masked_fill_(
            torch.arange(sk, device=DEV)[None, :] > torch.arange(sk - sq, sk, device=DEV)[:, None],
            -math.inf)
    elif case["mask"] == "padding":  # each sequence's own number of keys
        lens = torch.randint(1 + sk // 2, sk + 1, (b,), generator=g, device=DEV)
        mask = torch.zeros(b, 1, 1, sk, device=DEV).masked_fill_(
            torch.arange(sk, device=DEV)[None, None, None, :] >= lens[:, None, None, None],
            -math.inf)
    return q, k, v, mask


def _hybrid_config(case):
    return rx.Qwen35Config(max_batch=case["batch"], max_seq=case["tokens"])


def _hybrid_shapes(c):
    """The 0.8B model's parameters: path -> shape; 2-D ".weight"s of ``Q`` are W8."""
    root, out = "model.language_model.", {}
    width = c.linear_heads * c.linear_head_dim
    out[root + "embed_tokens"] = (c.vocab, c.hidden)
    for i, kind in enumerate(c.kinds()):
        p = f"{root}layers.{i}."
        if kind:
            a, d = p + "self_attn.", c.head_dim
            out[a + "q_proj"] = (c.heads * 2 * d, c.hidden)
            out[a + "k_proj"] = out[a + "v_proj"] = (c.kv_heads * d, c.hidden)
            out[a + "o_proj"] = (c.hidden, c.heads * d)
        else:
            a = p + "linear_attn."
            out[a + "in_proj_qkv"] = (3 * width, c.hidden)
            out[a + "in_proj_z"] = (width, c.hidden)
            out[a + "in_proj_b"] = out[a + "in_proj_a"] = (c.linear_heads, c.hidden)
            out[a + "out_proj"] = (c.hidden, width)
        out[p + "mlp.gate_proj"] = out[p + "mlp.up_proj"] = (c.intermediate, c.hidden)
        out[p + "mlp.down_proj"] = (c.hidden, c.intermediate)
    return out


def _hybrid_inputs(case, seed):
    g, c = _gen(seed), _hybrid_config(case)
    p = {}
    for path, (n, k) in _hybrid_shapes(c).items():
        p[path + ".weight"], p[path + ".scale"] = _codes(g, n, k, c.group)
    root, width = "model.language_model.", c.linear_heads * c.linear_head_dim
    for i, kind in enumerate(c.kinds()):
        pre = f"{root}layers.{i}."
        for name in ("input_layernorm", "post_attention_layernorm"):
            p[pre + name + ".weight"] = _normal(g, c.hidden, std=0.1)
        if kind:
            p[pre + "self_attn.q_norm.weight"] = _normal(g, c.head_dim, std=0.1)
            p[pre + "self_attn.k_norm.weight"] = _normal(g, c.head_dim, std=0.1)
        else:
            a = pre + "linear_attn."
            p[a + "conv1d.weight"] = _normal(g, 3 * width, 1, c.conv_kernel, std=0.5)
            p[a + "A_log"] = _normal(g, c.linear_heads, std=0.5)
            p[a + "dt_bias"] = _normal(g, c.linear_heads, std=0.5)
            p[a + "norm.weight"] = 1 + _normal(g, c.linear_head_dim, std=0.1)
    p[root + "norm.weight"] = _normal(g, c.hidden, std=0.1)
    ids = torch.randint(0, c.vocab, (case["batch"], case["tokens"]), generator=g, device=DEV,
                        dtype=torch.int32)
    return p, ids


def _decoder_config(case):
    return rx.DecoderConfig(layers=case["layers"], max_batch=case["batch"],
                            max_seq=case["prompt"] + case["steps"])


def _decoder_inputs(case, seed):
    g, c = _gen(seed), _decoder_config(case)
    p, d = {}, c.head_dim
    p["embed_tokens.weight"] = _normal(g, c.vocab, c.hidden).bfloat16()
    p["norm.weight"] = 1 + _normal(g, c.hidden, std=0.1)
    for i in range(c.layers):
        pre = f"layers.{i}."
        for name, n, k in (("self_attn.qkv_proj", (c.q_heads + 2 * c.kv_heads) * d, c.hidden),
                           ("self_attn.o_proj", c.hidden, c.q_heads * d),
                           ("mlp.gate_up_proj", 2 * c.intermediate, c.hidden),
                           ("mlp.down_proj", c.hidden, c.intermediate)):
            p[pre + name + ".weight"], p[pre + name + ".scale"] = _codes(g, n, k, 0)
        for name in ("input_layernorm", "post_attention_layernorm"):
            p[pre + name + ".weight"] = 1 + _normal(g, c.hidden, std=0.1)
        for name in ("q_norm", "k_norm"):
            p[pre + "self_attn." + name + ".weight"] = 1 + _normal(g, d, std=0.1)
    ids = torch.randint(0, c.vocab, (case["batch"], case["prompt"] + case["steps"]), generator=g,
                        device=DEV, dtype=torch.int32)
    return p, ids


# ---- one pass -------------------------------------------------------------------

def prepare(case, seed):
    rt, kind = _runtime(), case["kind"]
    wrap = rt.wrap_tensor
    state = {"case": case}
    if kind in ("linear", "head"):
        if kind == "linear":
            x, w, s = _linear_inputs(case, seed)
            out = torch.float32 if case["compute"] == "f32" else _FLOAT[case["x"]]
        else:
            (x, w), s, out = _head_inputs(case, seed), None, torch.float32
        torch.cuda.synchronize()
        wb = wrap(w)
        if case["packed"]:
            wb = rx.pack_weight(rt, wb)
            rt.synchronize()
        else:
            state["w"] = w
        y = torch.empty(case["rows"], case["n"], dtype=out, device=DEV)
        state.update(x=x, s=s, y=y, xb=wrap(x), wb=wb, sb=None if s is None else wrap(s),
                     yb=wrap(y), dtype=rx.DType.F32 if case.get("compute") == "f32" else rx.DType.BF16)
    elif kind in ("decode", "prefill", "masked"):
        q, k, v, extra = {"decode": _decode_inputs, "prefill": _prefill_inputs,
                          "masked": _masked_inputs}[kind](case, seed)
        y = torch.empty_like(q)
        state.update(t=(q, k, v, extra), y=y, yb=wrap(y),
                     b=[None if t is None else wrap(t) for t in (q, k, v, extra)])
    elif kind == "hybrid":
        p, ids = _hybrid_inputs(case, seed)
        torch.cuda.synchronize()
        model = rx.Qwen35Model(rt, _hybrid_config(case)).compile()
        model.bind_parameters({path: wrap(t) for path, t in p.items()})
        y = torch.empty(case["batch"], case["tokens"], model.cfg.vocab, device=DEV)
        state.update(p=p, ids=ids, y=y, model=model, idb=wrap(ids), yb=wrap(y))
    else:
        p, ids = _decoder_inputs(case, seed)
        torch.cuda.synchronize()
        model = rx.DecoderModel(rt, _decoder_config(case)).compile()
        model.bind_parameters({path: wrap(t) for path, t in p.items()})
        pieces = [ids[:, :case["prompt"]].contiguous()]
        pieces += [ids[:, case["prompt"] + i:][:, :1].contiguous() for i in range(case["steps"])]
        ys = [torch.empty(case["batch"], model.cfg.vocab, device=DEV) for _ in pieces]
        nxt = torch.empty(case["batch"], dtype=torch.int32, device=DEV)
        state.update(p=p, ids=pieces, ys=ys, nxt=nxt, model=model, nb=wrap(nxt),
                     calls=[(wrap(i), wrap(y)) for i, y in zip(pieces, ys)])
    torch.cuda.synchronize()
    return state


def run(state):
    rt, kind = _runtime(), state["case"]["kind"]
    if kind == "linear":
        rx.quantized_linear(rt, state["xb"], state["wb"], state["sb"], state["dtype"],
                            out=state["yb"])
        return state["y"]
    if kind == "head":
        rx.linear_bf16(rt, state["xb"], state["wb"], out=state["yb"])
        return state["y"]
    if kind == "decode":
        q, k, v, lens = state["b"]
        rx.grouped_query_attention(rt, q, k, v, lens, out=state["yb"])
        return state["y"]
    if kind == "prefill":
        q, k, v, starts = state["b"]
        rx.grouped_query_attention_prefill(rt, q, k, v, starts, out=state["yb"])
        return state["y"]
    if kind == "masked":
        q, k, v, mask = state["b"]
        rx.gqa_attention(rt, q, k, v, mask, out=state["yb"])
        return state["y"]
    if kind == "hybrid":
        state["model"].forward(state["idb"], state["yb"])
        return state["y"]
    model = state["model"]
    model.reset()
    for ids, logits in state["calls"]:
        model.forward(ids, logits, state["nb"])
    return state["ys"]


# ---- what a pass cannot do without ------------------------------------------------

_SIZE = {"bf16": 2, "f32": 4}


def _hybrid_work(case):
    c = _hybrid_config(case)
    t = case["batch"] * case["tokens"]
    shapes = _hybrid_shapes(c)
    weights = sum(n * k for n, k in shapes.values())
    scales = weights // c.group * 4
    flops = 2 * t * weights  # every projection and the tied head
    pairs = case["batch"] * case["tokens"] * (case["tokens"] + 1) // 2
    kinds = c.kinds()
    flops += sum(kinds) * 4 * pairs * c.heads * c.head_dim
    # per position and head: S k, S q and the rank-one update of a Dl x Dl state
    flops += (len(kinds) - sum(kinds)) * t * c.linear_heads * 6 * c.linear_head_dim ** 2
    return {"bytes": weights + scales + 4 * t + 4 * t * c.vocab, "flops": flops}


def _decoder_work(case):
    c = _decoder_config(case)
    b, s, steps = case["batch"], case["prompt"], case["steps"]
    d, hq, hkv = c.head_dim, c.q_heads, c.kv_heads
    layer = ((hq + 2 * hkv) * d * c.hidden + c.hidden * hq * d + 3 * c.hidden * c.intermediate)
    scales = 4 * ((hq + 2 * hkv) * d + 2 * c.hidden + 2 * c.intermediate)
    head = c.vocab * c.hidden
    kv = lambda length: 2 * 2 * b * length * hkv * d  # noqa: E731  bf16 keys and values
    nbytes = flops = 0
    for i in range(1 + steps):
        rows, seen = (b * s, s) if i == 0 else (b, s + i)
        nbytes += c.layers * (layer + scales + kv(seen)) + 2 * head + 4 * b * c.vocab
        flops += 2 * rows * c.layers * layer + 2 * b * head
        pairs = b * s * (s + 1) // 2 if i == 0 else b * seen
        flops += 4 * c.layers * pairs * hq * d
    return {"bytes": nbytes, "flops": flops}


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["rows"], case["n"], case["k"]
        out = 4 if case["compute"] == "f32" else _SIZE[case["x"]]
        nbytes = n * k + 4 * n * (k // (case["group"] or k)) + m * k * _SIZE[case["x"]] + m * n * out
        return {"bytes": nbytes, "flops": 2 * m * n * k}
    if kind == "head":
        m, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": 2 * n * k + 2 * m * k + 4 * m * n, "flops": 2 * m * n * k}
    if kind == "hybrid":
        return _hybrid_work(case)
    if kind == "decoder":
        return _decoder_work(case)
    b, hq, hkv, d = case["batch"], case["q_heads"], case["kv_heads"], case["dim"]
    if kind == "decode":  # the lengths' mean
        keys = b * (case["low"] + case["cap"]) // 2
        return {"bytes": 2 * keys * hkv * d * _SIZE[case["cache"]] + 2 * b * hq * d * _SIZE[case["q"]],
                "flops": 4 * keys * hq * d}
    if kind == "prefill":
        s, start = case["rows"], (case["start"] // 2 + case["start"]) // 2
        pairs = b * (s * start + s * (s + 1) // 2)
        return {"bytes": 2 * 2 * b * (start + s) * hkv * d + 2 * b * s * hq * d * _SIZE[case["q"]],
                "flops": 4 * pairs * hq * d}
    sq, sk = case["queries"], case["keys"]
    pairs = b * sq * sk
    if case["mask"] == "causal":
        pairs = b * (sq * (sk - sq) + sq * (sq + 1) // 2)
    elif case["mask"] == "padding":
        pairs = b * sq * (1 + sk // 2 + sk) // 2
    mask = {"causal": sq * sk, "padding": b * sk, "none": 0}[case["mask"]]
    return {"bytes": 4 * (2 * b * hkv * sk * d + 2 * b * hq * sq * d + mask), "flops": 4 * pairs * hq * d}


# ---- how far a correct implementation may be off ------------------------------------

# About four times the distance from ``exact`` measured on the listed and 30 drawn
# cases: results rounded to bf16 were 1.7e-3 (largest element 3.9e-3) away, f32 ones
# as noted. "max" is over the result's root mean square or the value, if larger.
_BF16 = {"rel": 6e-3, "max": 1.6e-2}


def tolerance(case):
    kind = case["kind"]
    if kind == "linear":
        # f32: codes times f32 rows split in two bf16 parts, 2.5e-6 (1.1e-5)
        return {"rel": 1e-5, "max": 5e-5} if case["compute"] == "f32" else _BF16
    if kind == "head":
        return _BF16
    if kind == "decode":  # f32: 2.6e-6 (2.2e-5)
        return {"rel": 1e-5, "max": 1e-4} if case["q"] == "f32" else _BF16
    if kind == "prefill":
        if case["dim"] == 128:  # probabilities rounded to bf16: 2.3e-3 (1.5e-2)
            return {"rel": 1e-2, "max": 6e-2}
        return {"rel": 1e-5, "max": 1e-4} if case["q"] == "f32" else _BF16
    if kind == "masked":  # 5.6e-7 (9.3e-6)
        return {"rel": 5e-6, "max": 5e-5}
    if kind == "hybrid":  # 24 layers of f32 sums: 8.9e-5 (6.3e-4)
        return {"rel": 4e-4, "max": 2.5e-3}
    return {"rel": 3e-2, "max": 0.16}  # four layers of bf16 results: 8.2e-3 (3.9e-2)


# ---- the same in 64 bits ------------------------------------------------------------

def _attend(q, k, v, mask=None):
    """q [Hq, Sq, D], k / v [Hkv, Sk, D], all f64; mask broadcast to [Hq, Sq, Sk]."""
    group = q.shape[0] // k.shape[0]
    out = torch.empty(q.shape[:2] + v.shape[-1:], dtype=torch.float64, device=q.device)
    for h in range(q.shape[0]):
        s = q[h] @ k[h // group].T / math.sqrt(q.shape[-1])
        if mask is not None:
            s = s + mask[min(h, mask.shape[0] - 1)]
        out[h] = torch.softmax(s, dim=-1) @ v[h // group]
    return out


def _causal(sq, sk, start):
    i = torch.arange(sq, device=DEV)[:, None] + start
    return torch.zeros(1, sq, sk, dtype=torch.float64, device=DEV).masked_fill_(
        (torch.arange(sk, device=DEV)[None, :] > i)[None], -math.inf)


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _rope(x, theta, width):
    """x [B, S, H, D]: split-half rotation of the first `width` dims."""
    half = width // 2
    freq = theta ** (-torch.arange(half, dtype=torch.float64, device=DEV) * 2 / width)
    angle = torch.arange(x.shape[1], dtype=torch.float64, device=DEV)[:, None] * freq
    c, s = angle.cos()[:, None], angle.sin()[:, None]
    a, b = x[..., :half], x[..., half:width]
    return torch.cat([a * c - b * s, b * c + a * s, x[..., width:]], dim=-1)


def _exact_hybrid(case, seed):
    p, ids = _hybrid_inputs(case, seed)
    c, root = _hybrid_config(case), "model.language_model."
    b, s, hl, dl = case["batch"], case["tokens"], c.linear_heads, c.linear_head_dim
    width = hl * dl
    sig = torch.sigmoid

    def proj(x, path):
        return x @ _weights(p[path + ".weight"], p[path + ".scale"]).T

    def norm(x, path):
        return _rms(x, 1 + p[path + ".weight"].double(), c.eps)

    table = _weights(p[root + "embed_tokens.weight"], p[root + "embed_tokens.scale"])
    h = table[ids.long()]
    for i, kind in enumerate(c.kinds()):
        pre = f"{root}layers.{i}."
        x = norm(h, pre + "input_layernorm")
        if kind:
            a, d = pre + "self_attn.", c.head_dim
            qg = proj(x, a + "q_proj").reshape(b, s, c.heads, 2 * d)
            q = _rope(norm(qg[..., :d], a + "q_norm"), c.theta, c.rotary_dim)
            k = proj(x, a + "k_proj").reshape(b, s, c.kv_heads, d)
            k = _rope(norm(k, a + "k_norm"), c.theta, c.rotary_dim)
            v = proj(x, a + "v_proj").reshape(b, s, c.kv_heads, d)
            o = torch.stack([_attend(q[j].transpose(0, 1), k[j].transpose(0, 1),
                                     v[j].transpose(0, 1), _causal(s, s, 0)) for j in range(b)])
            o = o.transpose(1, 2).reshape(b, s, -1) * sig(qg[..., d:].reshape(b, s, -1))
            h = h + proj(o, a + "o_proj")
        else:
            a = pre + "linear_attn."
            m = proj(x, a + "in_proj_qkv")
            taps = p[a + "conv1d.weight"].double().reshape(3 * width, -1)
            pad = torch.cat([m.new_zeros(b, taps.shape[1] - 1, 3 * width), m], dim=1)
            m = sum(pad[:, j:j + s] * taps[:, j] for j in range(taps.shape[1]))
            m = (m * sig(m)).reshape(b, s, 3, hl, dl)
            unit = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
            q, k, v = unit(m[:, :, 0]) / math.sqrt(dl), unit(m[:, :, 1]), m[:, :, 2]
            z = proj(x, a + "in_proj_z").reshape(b, s, hl, dl)
            beta = sig(proj(x, a + "in_proj_b"))
            g = proj(x, a + "in_proj_a") + p[a + "dt_bias"].double()
            g = torch.exp(-torch.nn.functional.softplus(g, threshold=200) * p[a + "A_log"].double().exp())
            state = m.new_zeros(b, hl, dl, dl)
            o = torch.empty_like(v)
            for t in range(s):
                state = state * g[:, t, :, None, None]
                seen = (k[:, t, :, None] @ state)[..., 0, :]
                delta = (v[:, t] - seen) * beta[:, t, :, None]
                state = state + k[:, t, :, :, None] * delta[..., None, :]
                o[:, t] = (q[:, t, :, None] @ state)[..., 0, :]
            o = _rms(o, p[a + "norm.weight"].double(), c.eps) * (z * sig(z))
            h = h + proj(o.reshape(b, s, width), a + "out_proj")
        x = norm(h, pre + "post_attention_layernorm")
        gate = proj(x, pre + "mlp.gate_proj")
        h = h + proj(gate * sig(gate) * proj(x, pre + "mlp.up_proj"), pre + "mlp.down_proj")
    return norm(h, root + "norm") @ table.T


def _exact_decoder(case, seed):
    p, ids = _decoder_inputs(case, seed)
    c = _decoder_config(case)
    b, s, d = case["batch"], case["prompt"] + case["steps"], c.head_dim

    def proj(x, path):
        return x @ _weights(p[path + ".weight"], p[path + ".scale"]).T

    def norm(x, path):
        return _rms(x, p[path + ".weight"].double(), c.eps)

    h = p["embed_tokens.weight"][ids.long()].double()
    for i in range(c.layers):
        pre = f"layers.{i}."
        x = proj(norm(h, pre + "input_layernorm"), pre + "self_attn.qkv_proj")
        q, k, v = x.reshape(b, s, -1, d).split([c.q_heads, c.kv_heads, c.kv_heads], dim=2)
        q = _rope(norm(q, pre + "self_attn.q_norm"), c.theta, d)
        k = _rope(norm(k, pre + "self_attn.k_norm"), c.theta, d)
        o = torch.stack([_attend(q[j].transpose(0, 1), k[j].transpose(0, 1), v[j].transpose(0, 1),
                                 _causal(s, s, 0)) for j in range(b)])
        h = h + proj(o.transpose(1, 2).reshape(b, s, -1), pre + "self_attn.o_proj")
        x = proj(norm(h, pre + "post_attention_layernorm"), pre + "mlp.gate_up_proj")
        gate, up = x.chunk(2, dim=-1)
        h = h + proj(gate * torch.sigmoid(gate) * up, pre + "mlp.down_proj")
    x = norm(h[:, case["prompt"] - 1:], "norm") @ p["embed_tokens.weight"].double().T
    return [x[:, i] for i in range(1 + case["steps"])]


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        x, u8, s = _linear_inputs(case, seed)
        w = _weights(u8, s)
        if case["compute"] == "bf16":  # the products' operands are bf16 by definition
            x, w = x.bfloat16(), _weights(u8, s, torch.float32).bfloat16()
        return x.double() @ w.double().T
    if kind == "head":
        x, w = _head_inputs(case, seed)
        return x.double() @ w.double().T
    if kind == "hybrid":
        return _exact_hybrid(case, seed)
    if kind == "decoder":
        return _exact_decoder(case, seed)
    if kind == "decode":
        q, k, v, lens = _decode_inputs(case, seed)
        rows = [_attend(q[i].double()[:, None], k[i, :, :n].double(), v[i, :, :n].double())[:, 0]
                for i, n in enumerate(lens.tolist())]
        return torch.stack(rows)
    if kind == "prefill":
        q, k, v, starts = _prefill_inputs(case, seed)
        rows = [_attend(q[i].double().transpose(0, 1), k[i].double(), v[i].double(),
                        _causal(q.shape[1], k.shape[2], n)).transpose(0, 1)
                for i, n in enumerate(starts.tolist())]
        return torch.stack(rows)
    q, k, v, mask = _masked_inputs(case, seed)
    rows = []
    for i in range(q.shape[0]):
        m = None
        if mask is not None:
            m = mask.double().reshape(1, *mask.shape) if mask.dim() == 2 else mask[i].double()
        rows.append(_attend(q[i].double(), k[i].double(), v[i].double(), m))
    return torch.stack(rows)
