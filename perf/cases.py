"""The workloads that this framework's performance is judged by: one GRPO iteration's
GPU work, call by call, through the entry points a program uses.

* ``attention``: the low-level decode loop's append + paged GQA attention.
* ``lora_decode``: the q/k/v/o NF4 + LoRA projections of a decode batch (no gradients).
* ``lora_train``: the same four projections forward and backward, as the policy update
  runs them (gradients of the input and of every adapter).
* ``mlp_train``: the frozen NF4 MLP (gate, up, SiLU, down) forward and backward.
* ``prefill``: a prompt cached through the model's layers (the KV cache comes back).
* ``decode``: one decode step of a model over a ragged batch (logits and KV cache).
* ``sample``: the top-p draw over a whole vocabulary.

Model shapes are those of the repository's configurations (Qwen2-1.5B and Qwen2-7B)
with fewer layers; every layer runs at its real size.
"""

from __future__ import annotations

import math
import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.getcwd(), "grpo-training-engine_amd"))

BS = 16    # KV block size
QB = 64    # NF4 blocksize
SHAPES = {  # hidden, MLP, query heads, KV heads, vocabulary
    "1.5b": (1536, 8960, 12, 2, 151936),
    "7b": (3584, 18944, 28, 4, 152064),
}


# ------------------------------------------------------------------ cases --

def listed():
    return [
        # one layer's attention of a small ragged group (the micro-batch of 4)
        dict(name="attention_group4", kind="attention", rows=4, heads=12, kv_heads=2,
             ctx_lo=512, ctx_hi=1024),
        # ... and of a large group with long contexts
        dict(name="attention_group64", kind="attention", rows=64, heads=28, kv_heads=4,
             ctx_lo=1024, ctx_hi=4096),
        # a decode batch's projections, called one by one
        dict(name="lora_decode_8", kind="lora_decode", rows=8, hidden=1536, kv=256, rank=16),
        # the policy update on a micro-batch of 4 short sequences
        dict(name="lora_train_256", kind="lora_train", batch=4, seq=64, hidden=1024, kv=256,
             rank=16, dtype="bf16", nested=False),
        # ... of 4 sequences of prompt + response, of no round length
        dict(name="lora_train_2092", kind="lora_train", batch=4, seq=523, hidden=1536, kv=256,
             rank=16, dtype="bf16", nested=False),
        # ... of a whole group of 8 at the larger model, double-quantized scales
        dict(name="lora_train_8192", kind="lora_train", batch=8, seq=1024, hidden=3584, kv=512,
             rank=16, dtype="bf16", nested=True),
        # ... in float16 with a smaller rank
        dict(name="lora_train_f16", kind="lora_train", batch=2, seq=331, hidden=1536, kv=256,
             rank=8, dtype="f16", nested=False),
        # the frozen MLP of the policy update
        dict(name="mlp_train_1024", kind="mlp_train", batch=2, seq=512, hidden=1536, inter=8960),
        # a 512-token prompt (its last token is the first decode step's input)
        dict(name="prefill_511", kind="prefill", shape="1.5b", layers=4, tokens=511),
        # one step of a group of 8 after a 512-token prompt
        dict(name="decode_8", kind="decode", shape="1.5b", layers=4, rows=8, ctx_lo=512,
             ctx_hi=1024),
        # one step of 64 rows of the larger model over long contexts
        dict(name="decode_64", kind="decode", shape="7b", layers=2, rows=64, ctx_lo=1024,
             ctx_hi=4096),
        # the trainer's default sampling (T 0.7, top-p 0.9) of a group of 8
        dict(name="sample_8", kind="sample", rows=8, vocab=151936, temperature=0.7, top_p=0.9,
             std=2.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attention", "lora_decode", "lora_train", "lora_train", "lora_train",
                       "mlp_train", "prefill", "decode", "sample"])
    if kind == "attention":
        kv = rng.choice([1, 2, 4])
        lo = _log_int(rng, 17, 2048)
        return dict(kind=kind, rows=_log_int(rng, 1, 64), heads=kv * rng.randint(1, 7),
                    kv_heads=kv, ctx_lo=lo, ctx_hi=min(4096, lo + _log_int(rng, 16, 2048)))
    if kind == "lora_decode":
        return dict(kind=kind, rows=_log_int(rng, 1, 64), hidden=128 * rng.randint(4, 28),
                    kv=128 * rng.choice([1, 2, 4]), rank=rng.choice([8, 16, 32]))
    if kind == "lora_train":
        batch = rng.randint(1, 8)
        return dict(kind=kind, batch=batch, seq=_log_int(rng, 16, 1024),
                    hidden=128 * rng.randint(4, 28), kv=128 * rng.choice([1, 2, 4]),
                    rank=rng.choice([8, 16, 16, 32]),
                    dtype=rng.choice(["bf16", "bf16", "bf16", "f16"]),
                    nested=rng.random() < 0.5)
    if kind == "mlp_train":
        return dict(kind=kind, batch=rng.randint(1, 4), seq=_log_int(rng, 16, 700),
                    hidden=128 * rng.randint(4, 16), inter=128 * rng.randint(8, 72))
    if kind == "prefill":
        return dict(kind=kind, shape="1.5b", layers=rng.randint(2, 4),
                    tokens=_log_int(rng, 17, 1400))
    if kind == "decode":
        lo = _log_int(rng, 32, 1024)
        return dict(kind=kind, shape="1.5b", layers=rng.randint(2, 4), rows=_log_int(rng, 1, 48),
                    ctx_lo=lo, ctx_hi=lo + _log_int(rng, 16, 1024))
    return dict(kind=kind, rows=_log_int(rng, 1, 32), vocab=151936,
                temperature=rng.choice([0.7, 1.0]), top_p=rng.choice([0.5, 0.9, 0.95]),
                std=rng.choice([0.03, 1.0, 2.0, 6.0]))


# ----------------------------------------------------------------- inputs --

NF4 = (-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453,
       -0.28444138169288635, -0.18477343022823334, -0.09105003625154495, 0.0,
       0.07958029955625534, 0.16093020141124725, 0.24611230194568634, 0.33791524171829224,
       0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape, std=1.0, dtype=torch.bfloat16):
    return (torch.randn(*shape, generator=g, device="cuda") * std).to(dtype)


def _nf4(g, n, k, std=0.02):
    """Packed bytes and float32 absmax of a random [n, k] weight, quantized to NF4."""
    blocks = (torch.randn(n * k // QB, QB, generator=g, device="cuda") * std)
    absmax = blocks.abs().amax(1)
    code = torch.tensor(NF4, device="cuda")
    q = torch.bucketize(blocks / absmax[:, None], (code[1:] + code[:-1]) / 2).to(torch.uint8)
    q = q.view(-1)
    return ((q[0::2] << 4) | q[1::2]), absmax


def _nested(absmax):
    """Double quantization of absmax: uint8 codes, codebook, scales of 256, offset."""
    offset = float(absmax.mean())
    pad = -absmax.numel() % 256
    d = F.pad(absmax - offset, (0, pad)).view(-1, 256)
    s2 = d.abs().amax(1)
    code2 = torch.linspace(-1.0, 1.0, 256, device="cuda")
    q = torch.bucketize(d / s2[:, None], (code2[1:] + code2[:-1]) / 2).to(torch.uint8)
    return q.view(-1)[:absmax.numel()].contiguous(), code2, s2, offset


def _unpack(packed, absmax, n, k, dtype):
    """[n, k] in float64: the values of the weight in the compute type."""
    b = packed.view(-1).long()
    q = torch.stack([b >> 4, b & 15], 1).view(-1, QB)
    code = torch.tensor(NF4, device="cuda")
    return (code[q] * absmax.view(-1, 1)).to(dtype).view(n, k).double()


DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}


def _lora_parts(c, seed):
    """Weights and inputs of the four projections, in the order q, k, v, o."""
    g = _gen(seed)
    h, kv, r, dt = c["hidden"], c["kv"], c["rank"], DTYPES[c.get("dtype", "bf16")]
    parts = []
    for name, n in (("q", h), ("k", kv), ("v", kv), ("o", h)):
        packed, absmax = _nf4(g, n, h)
        nested = _nested(absmax) if c.get("nested") else None
        parts.append(dict(name=name, n=n, packed=packed, absmax=absmax, nested=nested,
                          bias=None if name == "o" else _randn(g, n, std=0.02, dtype=dt),
                          a=_randn(g, r, h, std=0.01, dtype=dt),
                          b=_randn(g, n, r, std=0.01, dtype=dt)))
    lead = (1, c["rows"]) if "rows" in c else (c["batch"], c["seq"])
    x = _randn(g, *lead, h, dtype=dt)
    ao = _randn(g, *lead, h, std=0.5, dtype=dt)
    grads = [_randn(g, *lead, p["n"], std=0.1, dtype=dt) for p in parts]
    return parts, x, ao, grads


def _layer(p, hidden, rank, dtype):
    from grpo_mi355x.core.lora import ManualLoRALayer
    from grpo_mi355x.core.nf4 import Linear4bitNF4, Params4bit, QuantState

    base = Linear4bitNF4(hidden, p["n"], bias=p["bias"] is not None, device="cuda")
    code = torch.tensor(NF4, device="cuda")
    if p["nested"] is not None:
        q, code2, s2, offset = p["nested"]
        state = QuantState(q, (p["n"], hidden), code, QB, offset=offset,
                           state2=QuantState(s2, (s2.numel(),), code2, 256))
    else:
        state = QuantState(p["absmax"], (p["n"], hidden), code, QB)
    base.weight = Params4bit(p["packed"].view(-1, 1), state)
    layer = ManualLoRALayer(base, rank=rank, alpha=2 * rank).to("cuda").to(dtype)
    with torch.no_grad():
        if p["bias"] is not None:
            base.bias.copy_(p["bias"])
        layer.lora_A.weight.copy_(p["a"])
        layer.lora_B.weight.copy_(p["b"])
    return layer


def _tables(rows, need, width, seed):
    """Shuffled block tables [rows, width] (unused entries -1) over rows * width blocks."""
    perm = torch.randperm(rows * width, generator=torch.Generator().manual_seed(int(seed)))
    t = torch.full((rows, width), -1, dtype=torch.int32)
    at = 0
    for b, n in enumerate(need):
        t[b, :n] = perm[at:at + n].to(torch.int32)
        at += n
    return t


def _contexts(c, seed):
    """Tokens already cached, per row; no row is longer than the widest of the case."""
    g = torch.Generator().manual_seed(int(seed))
    lens = torch.randint(c["ctx_lo"], c["ctx_hi"], (c["rows"],), generator=g)
    return [int(v) for v in lens]


def _attention_inputs(c, seed):
    g = _gen(seed)
    ctx = _contexts(c, seed)
    width = -(-c["ctx_hi"] // BS)
    need = [-(-(n + 1) // BS) for n in ctx]
    shape = (c["rows"] * width, c["kv_heads"], BS, 128)
    return dict(ctx=ctx, k=_randn(g, *shape), v=_randn(g, *shape),
                tables=_tables(c["rows"], need, width, seed).cuda(),
                lens=torch.tensor(ctx, dtype=torch.int32, device="cuda"),
                q=_randn(g, c["rows"], c["heads"], 128),
                kn=_randn(g, c["rows"], c["kv_heads"], 128),
                vn=_randn(g, c["rows"], c["kv_heads"], 128))


def _fill_model(model, c, seed):
    """Seeded weights in every layer of the model (its embedding, norms and head are
    seeded by the model itself); returns them for exact()."""
    h, inter, hq, hkv, _ = SHAPES[c["shape"]]
    g = _gen(seed + 77)
    got = []
    for i in range(c["layers"]):
        w = dict(qkv=_nf4(g, (hq + 2 * hkv) * 128, h), o=_nf4(g, h, hq * 128),
                 gate_up=_nf4(g, 2 * inter, h), down=_nf4(g, h, inter),
                 lora=[(_randn(g, 16, k, std=0.01), _randn(g, n, 16, std=0.01)) for n, k in (
                     (hq * 128, h), (hkv * 128, h), (hkv * 128, h), (h, hq * 128))],
                 bias=[_randn(g, n * 128, std=0.02) for n in (hq, hkv, hkv)],
                 norms=[(1 + _randn(g, h, std=0.02).float()).bfloat16() for _ in range(2)])
        got.append(w)
        if model is None:
            continue
        layer = model.model.layers[i]
        at, mlp = layer.self_attn, layer.mlp
        with torch.no_grad():
            for st, key in ((at.qkv, "qkv"), (mlp.gate_up, "gate_up")):
                st.packed.copy_(w[key][0].view_as(st.packed))
                st.absmax.copy_(w[key][1].view_as(st.absmax))
            for lin, key in ((at.o_proj.base_layer, "o"), (mlp.down_proj, "down")):
                lin.weight.copy_(w[key][0].view_as(lin.weight))
                lin.weight.quant_state.absmax.copy_(w[key][1])
            for proj, (a, b) in zip((at.q_proj, at.k_proj, at.v_proj, at.o_proj), w["lora"]):
                proj.lora_A.weight.copy_(a)
                proj.lora_B.weight.copy_(b)
            for proj, b in zip((at.q_proj, at.k_proj, at.v_proj), w["bias"]):
                proj.base_layer.bias.copy_(b)
            layer.input_layernorm.weight.copy_(w["norms"][0])
            layer.post_attention_layernorm.weight.copy_(w["norms"][1])
    vocab = SHAPES[c["shape"]][4]
    top = dict(embed=_randn(g, vocab, h, std=0.02), head=_randn(g, vocab, h, std=0.02),
               norm=(1 + _randn(g, h, std=0.02).float()).bfloat16())
    if model is not None:
        with torch.no_grad():
            model.model.embed_tokens.weight.copy_(top["embed"])
            model.lm_head.weight.copy_(top["head"])
            model.model.norm.weight.copy_(top["norm"])
    return got, top


def _model(c, seed):
    from grpo_mi355x.rollout.qwen2 import Qwen2Config, build_random_model

    cfg = Qwen2Config.qwen2_7b() if c["shape"] == "7b" else Qwen2Config.qwen2_1_5b()
    cfg.num_hidden_layers = c["layers"]
    model = build_random_model(cfg, torch.device("cuda"), seed=int(seed))
    _fill_model(model, c, seed)
    return cfg, model


def _decode_inputs(c, seed):
    _, _, _, hkv, vocab = SHAPES[c["shape"]]
    ctx = _contexts(c, seed)
    need = [-(-(n + 1) // BS) for n in ctx]
    width = -(-(c["ctx_hi"] + BS) // BS)
    g = _gen(seed + 5)
    blocks = c["rows"] * width
    return dict(ctx=ctx, blocks=blocks, width=width,
                tables=_tables(c["rows"], need, width, seed).cuda(),
                tokens=torch.randint(0, vocab, (c["rows"],), generator=g, device="cuda"),
                kv=[[_randn(g, blocks, hkv, BS, 128) for _ in range(2)]
                    for _ in range(c["layers"])])


def _prompt(c, seed):
    return torch.randint(0, SHAPES[c["shape"]][4], (c["tokens"] + 1,),
                         generator=torch.Generator().manual_seed(int(seed)))


# ---------------------------------------------------------------- prepare --

def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "attention":
        s = _attention_inputs(c, seed)
        s["after"] = s["lens"] + 1
    elif kind in ("lora_decode", "lora_train"):
        parts, x, ao, grads = _lora_parts(c, seed)
        dt = DTYPES[c.get("dtype", "bf16")]
        s = dict(x=x, ao=ao, grads=grads,
                 layers=[_layer(p, c["hidden"], c["rank"], dt) for p in parts])
        if kind == "lora_train":
            s["x"].requires_grad_()
            s["ao"].requires_grad_()
    elif kind == "mlp_train":
        s = _mlp_inputs(c, seed)
        s["layers"] = [_plain_layer(*w) for w in s.pop("weights")]
        s["x"].requires_grad_()
    elif kind == "prefill":
        from grpo_mi355x.core.kv_pool import PagedKVPool
        from grpo_mi355x.rollout.decode import prefill_engine

        cfg, model = _model(c, seed)
        n = c["tokens"]
        blocks = -(-(n + 1) // BS)
        pool = PagedKVPool(cfg.num_hidden_layers, blocks, cfg.num_key_value_heads, cfg.head_dim,
                           BS, device="cuda")
        s = dict(pool=pool, n=n, prompt=_prompt(c, seed).cuda(),
                 table=_tables(1, [blocks], blocks, seed).cuda(),
                 engine=prefill_engine(model, pool, n, blocks))
        # a program's engine has cached other prompts before this one
        s["engine"].run_prompt(s["table"], torch.zeros_like(s["prompt"]), n)
    elif kind == "decode":
        from grpo_mi355x.core.kv_pool import PagedKVPool
        from grpo_mi355x.rollout.decode import DecodeEngine

        cfg, model = _model(c, seed)
        d = _decode_inputs(c, seed)
        pool = PagedKVPool(cfg.num_hidden_layers, d["blocks"], cfg.num_key_value_heads,
                           cfg.head_dim, BS, device="cuda")
        for i, (k, v) in enumerate(d.pop("kv")):
            pool.k[i].copy_(k)
            pool.v[i].copy_(v)
        eng = DecodeEngine(model, pool, c["rows"], d["width"], keep_logits=True)
        s = dict(engine=eng, pool=pool, batch=dict(
            tokens=d["tokens"], positions=torch.tensor(d["ctx"], device="cuda"),
            block_tables=d["tables"], limits=torch.full((c["rows"],), 16, device="cuda"),
            max_new_tokens=16))
        eng.start(**s["batch"])
        eng.capture()
    else:
        from grpo_mi355x import _lib

        lib = _lib.device_library()
        g = _gen(seed)
        m, v = c["rows"], c["vocab"]
        s = dict(lib=lib, check=_lib.check, stream=_lib.stream_handle,
                 logits=_randn(g, m, v, std=c["std"]),
                 draws=torch.randint(-2 ** 63, 2 ** 63 - 1, (m,), generator=g, device="cuda"),
                 tokens=torch.zeros(m, dtype=torch.int64, device="cuda"),
                 kept=torch.zeros(m, dtype=torch.int32, device="cuda"),
                 ws=torch.zeros(int(lib.grpo_sample_workspace_bytes(m, v)), dtype=torch.uint8,
                                device="cuda"))
    s["case"] = dict(c)
    return s


def _mlp_inputs(c, seed):
    g = _gen(seed)
    h, i = c["hidden"], c["inter"]
    weights = [(n, k, *_nf4(g, n, k)) for n, k in ((i, h), (i, h), (h, i))]
    return dict(weights=weights, x=_randn(g, c["batch"], c["seq"], h),
                grad=_randn(g, c["batch"], c["seq"], h, std=0.1))


def _plain_layer(n, k, packed, absmax):
    from grpo_mi355x.core.nf4 import Linear4bitNF4, Params4bit, QuantState

    lin = Linear4bitNF4(k, n, bias=False, device="cuda")
    lin.weight = Params4bit(packed.view(-1, 1),
                            QuantState(absmax, (n, k), torch.tensor(NF4, device="cuda"), QB))
    return lin


# -------------------------------------------------------------------- run --

def run(s):
    c, kind = s["case"], s["case"]["kind"]
    if kind == "attention":
        from grpo_mi355x.kernels import ops

        ops.paged_kv_append(s["kn"], s["vn"], s["k"], s["v"], s["tables"], s["lens"])
        out = ops.paged_attention_decode(s["q"], s["k"], s["v"], s["tables"], s["after"],
                                         1.0 / math.sqrt(128))
        return dict(out=out, k=s["k"], v=s["v"])
    if kind == "lora_decode":
        q, k, v, o = s["layers"]
        with torch.no_grad():
            return [q(s["x"]), k(s["x"]), v(s["x"]), o(s["ao"])]
    if kind == "lora_train":
        q, k, v, o = s["layers"]
        params = [p for m in s["layers"] for p in (m.lora_A.weight, m.lora_B.weight)]
        for t in params + [s["x"], s["ao"]]:
            t.grad = None
        ys = [q(s["x"]), k(s["x"]), v(s["x"]), o(s["ao"])]
        torch.autograd.backward(ys, s["grads"])
        return dict(y=[y.detach() for y in ys], x=s["x"].grad, ao=s["ao"].grad,
                    lora=[p.grad for p in params])
    if kind == "mlp_train":
        gate, up, down = s["layers"]
        s["x"].grad = None
        y = down(F.silu(gate(s["x"])) * up(s["x"]))
        y.backward(s["grad"])
        return dict(y=y.detach(), x=s["x"].grad)
    if kind == "prefill":
        s["engine"].run_prompt(s["table"], s["prompt"], s["n"])
        return dict(k=s["pool"].k, v=s["pool"].v)
    if kind == "decode":
        s["engine"].start(**s["batch"])
        s["engine"].step()
        return dict(logits=s["engine"].logits, k=s["pool"].k, v=s["pool"].v)
    m, v = s["logits"].shape
    s["check"](s["lib"].grpo_sample_top_p(
        s["logits"].data_ptr(), v, m, v, c["temperature"], c["top_p"], s["draws"].data_ptr(),
        s["tokens"].data_ptr(), s["kept"].data_ptr(), s["ws"].data_ptr(), s["ws"].numel(),
        s["stream"](s["logits"].device)), "sample_top_p")
    return dict(tokens=s["tokens"], kept=s["kept"])


# ------------------------------------------------------------------- work --

def _nf4_bytes(n, k):
    return n * k // 2 + n * k // QB * 4


def work(case):
    c, kind = case, case["kind"]
    if kind == "attention":
        mean = (c["ctx_lo"] + c["ctx_hi"]) / 2
        tok = c["rows"] * mean
        return dict(bytes=tok * c["kv_heads"] * 128 * 4 + c["rows"] * c["heads"] * 128 * 6
                    + tok / BS * 4, flops=4 * tok * c["heads"] * 128)
    if kind in ("lora_decode", "lora_train"):
        h, kv, r = c["hidden"], c["kv"], c["rank"]
        m = c["rows"] if kind == "lora_decode" else c["batch"] * c["seq"]
        outs = 2 * h + 2 * kv
        adapters = 4 * r * h + outs * r
        w = sum(_nf4_bytes(n, h) for n in (h, kv, kv, h)) + adapters * 2
        if kind == "lora_decode":
            return dict(bytes=w + 2 * m * h * 2 + m * outs * 2,
                        flops=2 * m * (outs * h + adapters))
        # forward: x, ao in, four outputs; backward: four gradients and x, ao in, the
        # gradients of x, ao and the adapters out
        return dict(bytes=2 * w + 2 * m * h * 2 + m * outs * 2 + m * outs * 2 + 2 * m * h * 2
                    + 2 * m * h * 2 + adapters * 2,
                    flops=2 * m * (2 * outs * h + 3 * adapters))
    if kind == "mlp_train":
        h, i, m = c["hidden"], c["inter"], c["batch"] * c["seq"]
        # forward keeps gate, up and act; backward reads them
        return dict(bytes=6 * _nf4_bytes(i, h) + 4 * m * h * 2 + 6 * m * i * 2,
                    flops=2 * 2 * 3 * m * i * h)
    h, inter, hq, hkv, vocab = SHAPES[c["shape"]] if "shape" in c else (0,) * 5
    if kind in ("prefill", "decode"):
        nqkv, layers = (hq + 2 * hkv) * 128, c["layers"]
        layer_w = (nqkv + hq * 128 + 3 * inter) * h
        layer_b = _nf4_bytes(1, layer_w) + (2 * (hq + 2 * hkv) * 128 + 5 * h) * 16 * 2
        if kind == "prefill":  # the last layer ends with its append
            n = c["tokens"]
            return dict(bytes=n * h * 2 + (layers - 1) * layer_b + _nf4_bytes(nqkv, h)
                        + layers * n * hkv * 128 * 4,
                        flops=2 * n * ((layers - 1) * layer_w + nqkv * h)
                        + (layers - 1) * 2 * n * n * hq * 128)
        m = c["rows"]
        tok = m * (c["ctx_lo"] + c["ctx_hi"]) / 2
        return dict(bytes=m * h * 2 + layers * (layer_b + tok * hkv * 128 * 4) + vocab * h * 2
                    + m * vocab * 2,
                    flops=2 * m * (layers * layer_w + vocab * h)
                    + layers * 4 * tok * hq * 128)
    return dict(bytes=c["rows"] * c["vocab"] * 2, flops=c["rows"] * c["vocab"] * 4)


def tolerance(case):
    kind = case["kind"]
    if kind == "sample":
        return "exact"
    if kind == "attention":  # float32 results of bf16 inputs
        return {"rel": 1e-5}
    if kind in ("lora_decode", "lora_train", "mlp_train"):
        # one rounding of each 16-bit intermediate and of the result
        return {"rel": 2e-3 if case.get("dtype") == "f16" else 1e-2}
    return {"rel": 0.02}  # 16-bit roundings of every layer, one after another


# ------------------------------------------------------------------ exact --

def _lora_exact(p, x, h, dt):
    """y of one projection and what its backward needs, in float64."""
    absmax = p["absmax"]
    if p["nested"] is not None:
        q, code2, s2, offset = p["nested"]
        absmax = (code2.double()[q.long()] * s2.double().repeat_interleave(256)[:q.numel()]
                  + torch.tensor(offset).double()).float()
    w = _unpack(p["packed"], absmax, p["n"], h, dt)
    a, b = p["a"].double(), p["b"].double()
    t = x @ a.t()
    y = x @ w.t() + 2.0 * (t @ b.t())
    return (y if p["bias"] is None else y + p["bias"].double()), w, a, b, t


def _rms(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6) * w.double()


def _rope(x, pos):
    """x [rows, heads, 128] rotated at pos [rows] (tables in bf16, as the model keeps them)."""
    inv = 1.0 / (1000000.0 ** (torch.arange(0, 128, 2, dtype=torch.int64).float() / 128)).cuda()
    f = pos.float()[:, None] * inv[None]
    f = torch.cat([f, f], -1)
    cos, sin = f.cos().bfloat16().double()[:, None], f.sin().bfloat16().double()[:, None]
    rot = torch.cat([-x[..., 64:], x[..., :64]], -1)
    return x * cos + rot * sin


def _layer_exact(w, h, pos, shape, attend):
    """One decoder layer; attend(q, k, v) -> attention output or None to stop after it."""
    hid, inter, hq, hkv, _ = shape
    bf = torch.bfloat16

    def linear(x, key, n, k, lora=None, bias=None):
        y = x @ _unpack(*w[key], n, k, bf).t()
        if bias is not None:
            y = y + bias
        if lora is not None:
            y = y + lora
        return y

    x = _rms(h, w["norms"][0])
    nq, nk = hq * 128, hkv * 128
    lo = torch.cat([2.0 * (x @ a.double().t()) @ b.double().t() for a, b in w["lora"][:3]], -1)
    qkv = linear(x, "qkv", nq + 2 * nk, hid, lo, torch.cat(w["bias"]).double())
    m = x.shape[0]
    q = _rope(qkv[:, :nq].reshape(m, hq, 128), pos)
    k = _rope(qkv[:, nq:nq + nk].reshape(m, hkv, 128), pos)
    v = qkv[:, nq + nk:].reshape(m, hkv, 128)
    o = attend(q, k, v)
    if o is None:
        return None
    o = o.reshape(m, nq)
    a, b = w["lora"][3]
    h = h + linear(o, "o", hid, nq, 2.0 * (o @ a.double().t()) @ b.double().t())
    x = _rms(h, w["norms"][1])
    gu = linear(x, "gate_up", 2 * inter, hid)
    act = F.silu(gu[:, :inter]) * gu[:, inter:]
    return h + linear(act, "down", hid, inter)


def _attend_row(q, k, v):
    """q [hq, 128], k and v [tokens, hkv, 128], float64."""
    rep = q.shape[0] // k.shape[1]
    k, v = k.repeat_interleave(rep, 1), v.repeat_interleave(rep, 1)
    s = (k * q[None]).sum(-1) / math.sqrt(128)
    return (torch.softmax(s, 0)[..., None] * v).sum(0)


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "sample":
        return None
    with torch.no_grad():
        if kind == "attention":
            d = _attention_inputs(c, seed)
            out = []
            for b, n in enumerate(d["ctx"]):
                blk = d["tables"][b, n // BS].long()
                d["k"][blk, :, n % BS] = d["kn"][b]
                d["v"][blk, :, n % BS] = d["vn"][b]
                t = d["tables"][b, :n // BS + 1].long()
                k, v = (d[z][t].transpose(1, 2).reshape(-1, c["kv_heads"], 128)[:n + 1].double()
                        for z in "kv")
                out.append(_attend_row(d["q"][b].double(), k, v))
            return dict(out=torch.stack(out), k=d["k"], v=d["v"])
        if kind in ("lora_decode", "lora_train"):
            parts, x, ao, grads = _lora_parts(c, seed)
            dt, h = DTYPES[c.get("dtype", "bf16")], c["hidden"]
            ys, lora, gx = [], [], {}
            for p, g in zip(parts, grads):
                src = ao if p["name"] == "o" else x
                xin = src.double().view(-1, h)
                y, w, a, b, t = _lora_exact(p, xin, h, dt)
                ys.append(y.view(*src.shape[:-1], p["n"]))
                if kind == "lora_train":
                    g = g.double().view(-1, p["n"])
                    gi = 2.0 * (g @ b)
                    key = "ao" if p["name"] == "o" else "x"
                    gx[key] = gx.get(key, 0) + (g @ w + gi @ a).view(src.shape)
                    lora += [gi.t().contiguous() @ xin, 2.0 * (g.t().contiguous() @ t)]
            return ys if kind == "lora_decode" else dict(y=ys, x=gx["x"], ao=gx["ao"], lora=lora)
        if kind == "mlp_train":
            d = _mlp_inputs(c, seed)
            wg, wu, wd = (_unpack(p, a, n, k, torch.bfloat16) for n, k, p, a in d["weights"])
            x, g = (d[z].double().view(-1, c["hidden"]) for z in ("x", "grad"))
            gate, up = x @ wg.t(), x @ wu.t()
            sg = torch.sigmoid(gate)
            y = (gate * sg * up) @ wd.t()
            ga = g @ wd
            gx = (ga * gate * sg) @ wu + (ga * up * sg * (1 + gate * (1 - sg))) @ wg
            return dict(y=y.view(d["x"].shape), x=gx.view(d["x"].shape))
        shape = SHAPES[c["shape"]]
        layers, top = _fill_model(None, c, seed)
        if kind == "prefill":
            n = c["tokens"]
            h = top["embed"][_prompt(c, seed)[:n].cuda()].double()
            pos = torch.arange(n, device="cuda")
            blocks = -(-(n + 1) // BS)
            table = _tables(1, [blocks], blocks, seed)[0].long().cuda()
            kc = torch.zeros(c["layers"], blocks, shape[3], BS, 128, dtype=torch.float64,
                             device="cuda")
            vc = torch.zeros_like(kc)
            mask = torch.full((n, n), -math.inf, dtype=torch.float64, device="cuda").triu(1)
            for i, w in enumerate(layers):
                def attend(q, k, v):
                    kc[i, table[pos // BS], :, pos % BS] = k
                    vc[i, table[pos // BS], :, pos % BS] = v
                    if i + 1 == c["layers"]:
                        return None
                    rep = shape[2] // shape[3]
                    kk, vv = (z.repeat_interleave(rep, 1).transpose(0, 1).contiguous()
                              for z in (k, v))
                    s = torch.matmul(q.transpose(0, 1).contiguous(),
                                     kk.transpose(1, 2).contiguous()) / math.sqrt(128) + mask
                    return torch.matmul(torch.softmax(s, -1), vv).transpose(0, 1)
                h = _layer_exact(w, h, pos, shape, attend)
            return dict(k=kc, v=vc)
        d = _decode_inputs(c, seed)
        h = top["embed"][d["tokens"]].double()
        pos = torch.tensor(d["ctx"], device="cuda")
        ks, vs = (torch.stack([kv[z] for kv in d["kv"]]).double() for z in (0, 1))
        for i, w in enumerate(layers):
            def attend(q, k, v):
                out = []
                for b, n in enumerate(d["ctx"]):
                    t = d["tables"][b, :n // BS + 1].long()
                    ks[i, t[-1], :, n % BS] = k[b]
                    vs[i, t[-1], :, n % BS] = v[b]
                    kr, vr = (z[i, t].transpose(1, 2).reshape(-1, shape[3], 128)[:n + 1]
                              for z in (ks, vs))
                    out.append(_attend_row(q[b], kr, vr))
                return torch.stack(out)
            h = _layer_exact(w, h, pos, shape, attend)
        head = _rms(h, top["norm"])
        logits = torch.cat([head @ z.double().t() for z in top["head"].split(32768)], -1)
        return dict(logits=logits, k=ks, v=vs)
