"""The measured workloads: what a program built on this package calls, over the sizes it calls them at.

Four kinds of work:

* ``linear``: one ``LowBitLinear`` on an activation, the building block of every converted model (module path);
* ``decode``: a few tokens of a running generation on the native engine (hipGraph steps, teacher-forced so that rounding
  cannot change which token comes next), with the step's logits;
* ``prefill``: a fresh prompt through the native engine: last-position logits and the key cache it leaves;
* ``train``: forward and backward of a LoRA adapter on a frozen low-bit linear (QLoRA fine-tuning).

The engine cases run a few layers of a model shape (a whole model repeats them) with its output head.  Weights are drawn
from a normal distribution and quantized here, in plain torch, into the checkpoint block layouts that the package loads.
"""
import math

import torch

DEV = "cuda"

# (hidden, intermediate, heads, kv heads, head dim, rope theta, experts): layer shapes the package's benchmark uses
SHAPES = {
    "tinyllama": (2048, 5632, 32, 4, 64, 1e4, 0),
    "llama2-7b": (4096, 11008, 32, 32, 128, 1e4, 0),
    "llama3-8b": (4096, 14336, 32, 8, 128, 5e5, 0),
    "mixtral-8x7b": (4096, 14336, 32, 8, 128, 1e6, 8),
}
VOCAB = 32000
EPS = 1e-5
TOP_K = 2
NF4 = (-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453, -0.28444138169288635, -0.18477343022823334,
       -0.09105003625154495, 0.0, 0.07958029955625534, 0.16093020141124725, 0.24611230194568634, 0.33791524171829224,
       0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0)
# bytes per element of a checkpoint block, elements per block
FORMATS = {"sym_int4": (18 / 32, 32), "asym_int4": (20 / 32, 32), "nf4": (34 / 64, 64), "sym_int8": (34 / 32, 32),
           "fp8_e5m2": (34 / 32, 32), "q4_k": (144 / 256, 256), "q6_k": (210 / 256, 256)}


def listed():
    return [
        # smallest call: one token through the attention output projection of a 1B model
        dict(name="linear 1x2048 sym_int4", kind="linear", rows=1, n=2048, k=2048, fmt="sym_int4", dtype="fp16"),
        # a token through a down projection of a GGUF Q4_K_M file, which keeps half of those in q6_k
        dict(name="linear 1x11008 q6_k", kind="linear", rows=1, n=4096, k=11008, fmt="q6_k", dtype="fp16"),
        # a short bf16 prompt through an 8-bit projection of ragged width
        dict(name="linear 203x4544 sym_int8", kind="linear", rows=203, n=4672, k=4544, fmt="sym_int8", dtype="bf16"),
        # a large batch of hidden states (embedding / evaluation jobs) through an nf4 projection
        dict(name="linear 3000x4096 nf4", kind="linear", rows=3000, n=14336, k=4096, fmt="nf4", dtype="bf16"),
        # chat with a small model just after a short prompt: nothing but latency
        dict(name="decode tinyllama b1", kind="decode", model="tinyllama", layers=8, batch=1, past=45, steps=8,
             fmt="sym_int4", kv="fp16"),
        # the package's headline: one sequence, 1024-token prompt, 8-bit cache
        dict(name="decode llama2-7b b1", kind="decode", model="llama2-7b", layers=4, batch=1, past=1024, steps=8,
             fmt="sym_int4", kv="fp8"),
        # a batch of sequences with a grouped-query model, GGUF 4-bit weights, 16-bit cache
        dict(name="decode llama3-8b b12", kind="decode", model="llama3-8b", layers=4, batch=12, past=1900, steps=4,
             fmt="q4_k", kv="fp16"),
        # a full serving batch
        dict(name="decode llama2-7b b64", kind="decode", model="llama2-7b", layers=3, batch=64, past=1000, steps=4,
             fmt="sym_int4", kv="fp8"),
        # a short question to a chat model
        dict(name="prefill llama3-8b 77", kind="prefill", model="llama3-8b", layers=4, batch=1, tokens=77, fmt="asym_int4"),
        # the headline's prompt
        dict(name="prefill llama2-7b 1024", kind="prefill", model="llama2-7b", layers=4, batch=1, tokens=1024, fmt="sym_int4"),
        # a long document
        dict(name="prefill llama3-8b 7700", kind="prefill", model="llama3-8b", layers=3, batch=1, tokens=7700, fmt="sym_int4"),
        # a QLoRA micro-batch of 4 x 256 tokens on a 70B projection (whose dense copies would not fit beside it)
        dict(name="train 1024x8192 nf4", kind="train", rows=1024, n=8192, k=8192, rank=8, fmt="nf4"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "decode", "decode", "decode", "prefill", "prefill", "train"])
    if kind == "linear":
        fmt = rng.choice(list(FORMATS))
        step = max(32, FORMATS[fmt][1])
        k = _log_int(rng, 1024, 14336) // step * step
        return dict(kind=kind, rows=_log_int(rng, 1, 4096), n=_log_int(rng, 1024, 14336), k=k, fmt=fmt,
                    dtype=rng.choice(["fp16", "bf16"]))
    if kind == "decode":
        batch = _log_int(rng, 1, 64)
        past = _log_int(rng, 20, min(4000, 65000 // batch))
        model = rng.choice(["tinyllama", "llama2-7b", "llama3-8b", "mixtral-8x7b" if batch <= 8 else "llama3-8b"])
        return dict(kind=kind, model=model, layers=1 if model == "mixtral-8x7b" else rng.randint(2, 4), batch=batch,
                    past=past, steps=4, fmt=rng.choice(["sym_int4", "sym_int4", "asym_int4", "nf4", "q4_k"]),
                    kv=rng.choice(["fp16", "fp8"]))
    if kind == "prefill":
        tokens = _log_int(rng, 20, 7700)
        return dict(kind=kind, model=rng.choice(["tinyllama", "llama2-7b", "llama3-8b"]), layers=rng.randint(2, 3),
                    batch=rng.choice([1, 1, 1, 2, 3]) if tokens < 2500 else 1, tokens=tokens,
                    fmt=rng.choice(["sym_int4", "sym_int4", "asym_int4", "nf4", "q4_k"]))
    return dict(kind=kind, rows=_log_int(rng, 64, 2048), n=rng.choice([1024, 2048, 4096, 5632, 8192, 11008]),
                k=rng.choice([2048, 4096, 8192]), rank=rng.choice([8, 8, 16]), fmt=rng.choice(["nf4", "sym_int4"]))


# ------------------------------------------------------------------------------------------------ weights
def _gen(seed, tag):
    g = torch.Generator(device=DEV)
    g.manual_seed((seed * 1000003 + tag * 7919 + 12345) % (1 << 62))
    return g


def _f16(x):
    return x.to(torch.float16)


def _weight(fmt, n, k, std, seed, tag):
    """Codes and scales of a normally distributed [n, k] matrix quantized to ``fmt``."""
    w = torch.randn(n, k, generator=_gen(seed, tag), device=DEV) * std
    if fmt == "q4_k":
        b = w.view(n, k // 256, 8, 32)
        lo, hi = b.amin(-1).clamp_max(0), b.amax(-1)
        sc, mn = (hi - lo) / 15, -lo
        d, dm = _f16(sc.amax(-1, keepdim=True) / 63), _f16(mn.amax(-1, keepdim=True) / 63)
        s6 = (sc / d.float().clamp_min(1e-12)).round().clamp(1, 63)
        m6 = (mn / dm.float().clamp_min(1e-12)).round().clamp(0, 63)
        q = ((b + (dm.float() * m6)[..., None]) / (d.float() * s6)[..., None]).round().clamp(0, 15)
        return dict(fmt=fmt, n=n, k=k, q=q.to(torch.uint8), d=d, m=dm, s=s6.to(torch.uint8), ms=m6.to(torch.uint8))
    if fmt == "q6_k":
        b = w.view(n, k // 256, 16, 16)
        sc = b.abs().amax(-1) / 31
        d = _f16(sc.amax(-1, keepdim=True) / 127)
        s8 = (sc / d.float().clamp_min(1e-12)).round().clamp(1, 127)
        q = (b / (d.float() * s8)[..., None]).round().clamp(-32, 31)
        return dict(fmt=fmt, n=n, k=k, q=(q + 32).to(torch.uint8), d=d, s=s8.to(torch.int8))
    qk = FORMATS[fmt][1]
    b = w.view(n, k // qk, qk)
    big = b.abs().amax(-1, keepdim=True)
    if fmt == "sym_int4":
        at = b.abs().argmax(-1, keepdim=True)
        d = _f16(b.gather(-1, at) / -8)
        q = (b / d.float()).round().add(8).clamp(0, 15).to(torch.uint8)
        return dict(fmt=fmt, n=n, k=k, q=q, d=d)
    if fmt == "asym_int4":
        lo, hi = b.amin(-1, keepdim=True), b.amax(-1, keepdim=True)
        d, m = _f16((hi - lo) / 15), _f16(lo)
        return dict(fmt=fmt, n=n, k=k, q=((b - m.float()) / d.float()).round().clamp(0, 15).to(torch.uint8), d=d, m=m)
    if fmt == "nf4":
        d = _f16(big)
        table = torch.tensor(NF4, device=DEV)
        q = torch.bucketize((b / d.float()).contiguous(), (table[1:] + table[:-1]) / 2)
        return dict(fmt=fmt, n=n, k=k, q=q.to(torch.uint8), d=d)
    if fmt == "sym_int8":
        d = _f16(big / 127)
        return dict(fmt=fmt, n=n, k=k, q=(b / d.float()).round().clamp(-127, 127).to(torch.int8), d=d)
    d = _f16(big / 57344)
    return dict(fmt=fmt, n=n, k=k, q=(b / d.float()).clamp(-57344, 57344).to(torch.float8_e5m2), d=d)


def _bytes(*parts):
    return torch.cat([p.contiguous().view(torch.uint8).flatten(1) for p in parts], 1)


def _pack(w):
    """The checkpoint's block bytes (on the host, as a loader holds them)."""
    fmt, q = w["fmt"], w["q"]
    if fmt in ("sym_int4", "asym_int4", "nf4"):
        h = q.shape[-1] // 2
        q2 = (q[..., :h] | (q[..., h:] << 4)).flatten(0, 1)
        heads = [w[x].flatten(0, 1) for x in ("d", "m") if x in w]
        return _bytes(*heads, q2).flatten().cpu()
    if fmt == "q4_k":
        q = q.flatten(0, 1).view(-1, 4, 2, 32)
        s, m = w["s"].flatten(0, 1), w["ms"].flatten(0, 1)
        packed = torch.cat([s[:, :4] | (s[:, 4:] >> 4 << 6), m[:, :4] | (m[:, 4:] >> 4 << 6),
                            (s[:, 4:] & 15) | ((m[:, 4:] & 15) << 4)], 1)
        return _bytes(w["d"].flatten(0, 1), w["m"].flatten(0, 1), packed, q[:, :, 0] | (q[:, :, 1] << 4)).flatten().cpu()
    if fmt == "q6_k":
        q = q.flatten(0, 1).view(-1, 2, 4, 32)           # halves of 128, quarters of 32
        lo, hi = q & 15, q >> 4
        ql = torch.cat([lo[:, :, 0] | (lo[:, :, 2] << 4), lo[:, :, 1] | (lo[:, :, 3] << 4)], 2)
        qh = hi[:, :, 0] | (hi[:, :, 1] << 2) | (hi[:, :, 2] << 4) | (hi[:, :, 3] << 6)
        return _bytes(ql, qh, w["s"].flatten(0, 1), w["d"].flatten(0, 1)).flatten().cpu()
    return _bytes(w["d"].flatten(0, 1), q.flatten(0, 1)).flatten().cpu()


def _dense(w):
    """float64 [n, k]"""
    fmt = w["fmt"]
    d = w["d"].double()
    if fmt == "q4_k":
        v = w["q"].double() * (d * w["s"].double())[..., None] - (w["m"].double() * w["ms"].double())[..., None]
    elif fmt == "q6_k":
        v = (w["q"].double() - 32) * (d * w["s"].double())[..., None]
    elif fmt == "sym_int4":
        v = (w["q"].double() - 8) * d
    elif fmt == "asym_int4":
        v = w["q"].double() * d + w["m"].double()
    elif fmt == "nf4":
        v = torch.tensor(NF4, device=DEV, dtype=torch.float32).double()[w["q"].int()] * d
    else:
        v = w["q"].double() * d
    return v.reshape(w["n"], w["k"])


def _params(fmt, n, k, std, seed, tag):
    from bigdl_amd import qtypes as Q
    from bigdl_amd.transformers.low_bit_linear import FP4Params
    return FP4Params(_pack(_weight(fmt, n, k, std, seed, tag)), quantized=True, _shape=(n, k), qtype=Q.ggml_tensor_qtype[fmt])


def _module(fmt, n, k, seed):
    from bigdl_amd import qtypes as Q
    from bigdl_amd.transformers.low_bit_linear import LowBitLinear
    m = LowBitLinear(k, n, Q.ggml_tensor_qtype[fmt], bias=False)
    m.weight = _params(fmt, n, k, k ** -0.5, seed, 1)
    return m.to(DEV)


def _dtype(case):
    return torch.bfloat16 if case["kind"] == "train" or case["dtype"] == "bf16" else torch.float16


def _activations(case, seed, rows, width, tag):
    return torch.randn(rows, width, generator=_gen(seed, tag), device=DEV).to(_dtype(case))


# ------------------------------------------------------------------------------------------------ engine cases
def _matrices(case):
    """(name, rows, columns, std) of a layer's matrices; experts are stacked by rows."""
    h, i, hq, hkv, d, _, e = SHAPES[case["model"]]
    out = h ** -0.5 / math.sqrt(2 * case["layers"])
    m = [("qkv", (hq + 2 * hkv) * d, h, h ** -0.5), ("o", h, hq * d, out)]
    x = max(1, e)
    return m + [("gate", x * i, h, h ** -0.5), ("up", x * i, h, h ** -0.5), ("down", x * h, i, i ** -0.5)]


def _small(case, seed):
    """embedding, norms and routers: (embed, [(input norm, post norm, router)], final norm)"""
    h, e = SHAPES[case["model"]][0], SHAPES[case["model"]][6]
    g = _gen(seed, 2)

    def norm():
        return _f16(1 + 0.02 * torch.randn(h, generator=g, device=DEV))

    embed = _f16(torch.randn(VOCAB, h, generator=g, device=DEV) * 0.5)
    layers = [(norm(), norm(), _f16(torch.randn(e, h, generator=g, device=DEV) * h ** -0.5) if e else None)
              for _ in range(case["layers"])]
    return embed, layers, norm()


def _tokens(case, seed):
    n = case["past"] + case["steps"] if case["kind"] == "decode" else case["tokens"]
    return torch.randint(0, VOCAB, (case["batch"], n), generator=_gen(seed, 3), device=DEV)


def _engine(case, seed):
    from bigdl_amd import qtypes as Q
    from bigdl_amd.models.decoder import DecoderConfig, LayerWeights, Lin, NativeDecoder
    from bigdl_amd.models.moe import MoEWeights
    h, i, hq, hkv, d, theta, e = SHAPES[case["model"]]
    cfg = DecoderConfig(vocab_size=VOCAB, hidden_size=h, intermediate_size=i, num_layers=case["layers"], num_heads=hq,
                        num_kv_heads=hkv, head_dim=d, rms_eps=EPS, rope_theta=theta, max_position=8192, num_experts=e,
                        top_k=TOP_K if e else 0, moe_intermediate_size=i if e else 0)
    fmt = case["fmt"]
    embed, small, final = _small(case, seed)
    layers = []
    for li, (n1, n2, router) in enumerate(small):
        p = {name: _params(fmt, n, k, std, seed, 100 + 10 * li + j).to(DEV)
             for j, (name, n, k, std) in enumerate(_matrices(case))}
        lw = LayerWeights(input_norm=n1, qkv=Lin(p["qkv"]), o=Lin(p["o"]), post_norm=n2)
        if e:
            lw.moe = MoEWeights(router, p["gate"].data, p["up"].data, p["down"].data, Q.ggml_tensor_qtype[fmt], e, TOP_K, h, i)
        else:
            lw.gate, lw.up, lw.down = Lin(p["gate"]), Lin(p["up"]), Lin(p["down"])
        layers.append(lw)
    head = Lin(_params(fmt, VOCAB, h, h ** -0.5, seed, 4).to(DEV))
    return NativeDecoder(cfg, embed, layers, final, head, device=DEV)


# ------------------------------------------------------------------------------------------------ the four functions
def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        return dict(kind=kind, lin=_module(case["fmt"], case["n"], case["k"], seed).eval(),
                    x=_activations(case, seed, case["rows"], case["k"], 5))
    if kind == "train":
        from bigdl_amd.transformers.qlora import LoraConfig, get_peft_model
        base = torch.nn.Module()
        base.proj = _module(case["fmt"], case["n"], case["k"], seed)
        model = get_peft_model(base, LoraConfig(r=case["rank"], lora_alpha=2 * case["rank"], target_modules=["proj"]))
        lora = model.get_base_model().proj.train()
        a, b = (next(iter(m.values())).weight for m in (lora.lora_A, lora.lora_B))
        wa, wb = _adapters(case, seed)
        with torch.no_grad():
            a.copy_(wa)
            b.copy_(wb)
        return dict(kind=kind, lora=lora, a=a, b=b, x=_activations(case, seed, case["rows"], case["k"], 5).requires_grad_(),
                    gy=_activations(case, seed, case["rows"], case["n"], 6))
    eng = _engine(case, seed)
    ids = _tokens(case, seed)
    if kind == "prefill":
        eng.ensure_cache(case["batch"], case["tokens"] + 128, fp8=False)
        return dict(kind=kind, eng=eng, ids=ids, layers=case["layers"])
    past = case["past"]
    eng.ensure_cache(case["batch"], past + case["steps"] + 32, fp8=case["kv"] == "fp8")
    eng.prefill(ids[:, :past])
    return dict(kind=kind, eng=eng, past=past, ids=[ids[:, past + j:past + j + 1].contiguous() for j in range(case["steps"])])


def run(state):
    kind = state["kind"]
    if kind == "linear":
        with torch.no_grad():
            return state["lin"](state["x"])
    if kind == "train":
        x, a, b = state["x"], state["a"], state["b"]
        x.grad = a.grad = b.grad = None
        y = state["lora"](x)
        y.backward(state["gy"])
        return [y.detach(), x.grad, a.grad, b.grad]
    eng = state["eng"]
    if kind == "prefill":
        eng.cache.reset()
        logits = eng.prefill(state["ids"])
        s = state["ids"].shape[1]
        return [logits] + [eng.cache.k[li][:, :, :s] for li in range(state["layers"])]
    eng.cache.crop(state["past"])
    return [eng.decode(ids, 1)[0].clone() for ids in state["ids"]]


def _adapters(case, seed):
    g = _gen(seed, 7)
    r = case["rank"]
    return tuple((torch.randn(*s, generator=g, device=DEV) * std).to(torch.bfloat16)
                 for s, std in (((r, case["k"]), case["k"] ** -0.5), ((case["n"], r), 0.05)))


def work(case):
    kind = case["kind"]
    if kind in ("linear", "train"):
        m, n, k = case["rows"], case["n"], case["k"]
        wb = n * k * FORMATS[case["fmt"]][0]
        if kind == "linear":
            return {"bytes": wb + 2 * m * (n + k), "flops": 2 * m * n * k}
        r = case["rank"]
        return {"bytes": 2 * wb + 2 * (2 * m * (n + k)) + 8 * r * (n + k), "flops": 4 * m * n * k + 10 * m * r * (n + k)}
    h, i, hq, hkv, d, _, e = SHAPES[case["model"]]
    b, layers, per = case["batch"], case["layers"], FORMATS[case["fmt"]][0]
    attn_w = h * (2 * hq + 2 * hkv) * d
    ffn = 3 * h * i
    if kind == "decode":
        kvb = 1 if case["kv"] == "fp8" else 2
        touched = min(e, b * TOP_K) if e else 1
        active = TOP_K if e else 1
        one_bytes = one_flops = 0
        for j in range(case["steps"]):
            keys = case["past"] + j + 1
            one_bytes += layers * ((attn_w + touched * ffn) * per + 2 * b * keys * hkv * d * kvb) + VOCAB * h * per + 4 * b * VOCAB
            one_flops += 2 * b * (layers * (attn_w + active * ffn + 2 * keys * hq * d) + VOCAB * h)
        return {"bytes": one_bytes, "flops": one_flops}
    s = case["tokens"]
    return {"bytes": layers * ((attn_w + ffn) * per + 4 * b * s * hkv * d) + VOCAB * h * per + 2 * b * s * h + 4 * b * VOCAB,
            "flops": 2 * b * (layers * (s * (attn_w + ffn) + s * (s + 1) * hq * d) + VOCAB * h)}


def tolerance(case):
    # each about four times what the path measures off its exact() result
    if case["kind"] == "linear":
        return {"rel": 7e-3 if case["dtype"] == "bf16" else 1.2e-3}
    if case["kind"] == "train":
        return {"rel": 0.012}
    if case["kind"] == "decode":
        # (a router's choice between two nearly equal experts, and a cached key's e5m2 code, can fall either way)
        return {"rel": 0.02, "max": 0.8} if case["model"].startswith("mixtral") else {"rel": 0.01}
    return {"rel": 8e-3}


# ------------------------------------------------------------------------------------------------ 64-bit results
def _norm(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x, theta):
    """x [b, s, heads, d], positions 0 .. s-1, halves rotated"""
    s, d = x.shape[1], x.shape[-1]
    inv = theta ** (-torch.arange(0, d, 2, dtype=torch.float64, device=DEV) / d)
    ang = torch.arange(s, dtype=torch.float64, device=DEV)[:, None, None] * inv
    c, sn = ang.cos(), ang.sin()
    x0, x1 = x[..., : d // 2], x[..., d // 2:]
    return torch.cat([x0 * c - x1 * sn, x1 * c + x0 * sn], -1)


def _byte(x):
    return x.to(torch.float16).to(torch.float8_e5m2).double()


def _attend(q, k, v, offset):
    """causal; q [b, hq, s, d] at positions offset .., k / v [b, hkv, t, d]"""
    g = q.shape[1] // k.shape[1]
    k, v = k.repeat_interleave(g, 1), v.repeat_interleave(g, 1)
    out = torch.empty_like(q)
    for r in range(0, q.shape[2], 1024):
        sc = q[:, :, r:r + 1024] @ k.transpose(-1, -2) / math.sqrt(q.shape[-1])
        pos = offset + torch.arange(r, r + sc.shape[2], device=DEV)
        sc.masked_fill_(torch.arange(k.shape[2], device=DEV)[None] > pos[:, None], -math.inf)
        out[:, :, r:r + 1024] = torch.softmax(sc, -1) @ v
    return out


def _model(case, seed):
    """logits of the wanted positions [b, wanted, V] and the rotated keys of every layer"""
    h, i, hq, hkv, d, theta, e = SHAPES[case["model"]]
    embed, small, final = _small(case, seed)
    ids = _tokens(case, seed)
    decode = case["kind"] == "decode"
    past = case["past"] if decode else ids.shape[1]
    fp8 = decode and case["kv"] == "fp8"
    x = embed[ids].double()
    b, s = ids.shape
    per = max(1, (1 << 13) // s)
    keys = []
    for li, (n1, n2, router) in enumerate(small):
        w = {name: _dense(_weight(case["fmt"], n, k, std, seed, 100 + 10 * li + j))
             for j, (name, n, k, std) in enumerate(_matrices(case))}
        kept = []
        for b0 in range(0, b, per):
            xb = x[b0:b0 + per]
            qkv = _norm(xb, n1) @ w["qkv"].t()
            q = _rope(qkv[..., : hq * d].unflatten(-1, (hq, d)), theta).transpose(1, 2)
            k = _rope(qkv[..., hq * d:(hq + hkv) * d].unflatten(-1, (hkv, d)), theta).transpose(1, 2)
            v = qkv[..., (hq + hkv) * d:].unflatten(-1, (hkv, d)).transpose(1, 2)
            a = torch.cat([torch.cat([_attend(q[j:j + 1, :, :past], k[j:j + 1, :, :past], v[j:j + 1, :, :past], 0)
                                      for j in range(q.shape[0])])]
                          + ([_attend(q[:, :, past:], _byte(k) if fp8 else k, _byte(v) if fp8 else v, past)] if decode else []), 2)
            if not decode:
                kept.append(k)
            xb = xb + a.transpose(1, 2).flatten(2) @ w["o"].t()
            y = _norm(xb, n2)
            if e:
                p, at = torch.softmax(y @ router.double().t(), -1).topk(TOP_K, -1)
                p = p / p.sum(-1, keepdim=True)
                out = torch.zeros_like(y)
                for j in range(e):
                    wg, wu, wd = (w[n][j * r:(j + 1) * r] for n, r in (("gate", i), ("up", i), ("down", h)))
                    share = (p * (at == j)).sum(-1)
                    here = share > 0
                    z = y[here]
                    out[here] += share[here][:, None] * ((torch.nn.functional.silu(z @ wg.t()) * (z @ wu.t())) @ wd.t())
                xb = xb + out
            else:
                xb = xb + (torch.nn.functional.silu(y @ w["gate"].t()) * (y @ w["up"].t())) @ w["down"].t()
            x[b0:b0 + per] = xb
        if kept:
            keys.append(torch.cat(kept))
        del w
    x = _norm(x[:, past:] if decode else x[:, -1:], final)
    return x @ _dense(_weight(case["fmt"], VOCAB, h, h ** -0.5, seed, 4)).t(), keys


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind in ("linear", "train"):
        w = _dense(_weight(case["fmt"], case["n"], case["k"], case["k"] ** -0.5, seed, 1))
        x = _activations(case, seed, case["rows"], case["k"], 5).double()
        if kind == "linear":
            return x @ w.t()
        gy = _activations(case, seed, case["rows"], case["n"], 6).double()
        a, b = (t.double() for t in _adapters(case, seed))
        scale = 2.0
        return [x @ w.t() + scale * (x @ a.t()) @ b.t(), gy @ w + scale * (gy @ b) @ a, scale * (gy @ b).t() @ x,
                scale * gy.t() @ (x @ a.t())]
    logits, keys = _model(case, seed)
    if kind == "prefill":
        return [logits] + keys
    return [logits[:, j] for j in range(case["steps"])]
