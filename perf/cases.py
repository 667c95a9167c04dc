"""The measured workloads of one rank's quantized inference path.

Every case is a call a serving program makes through the layer classes: a
quantized projection, an MLP, an attention layer (prefill and decode), a prefill
of a decoder from token ids to logits and one greedy decode step of a full decoder.
Shapes are those of the TinyLlama, Llama-3-8B and Llama-3-70B rank-0-of-8
configurations that bench.py and the tests use; ``draw`` spreads the row counts,
widths, lengths, batch sizes and code widths over the ranges between a single token
and a batch of long prompts.

Inputs are random: weights N(0, 0.02) quantized to the affine group-64 format (the
distribution of a trained projection's groups), activations N(0, 1) in bfloat16,
uniform token ids.
"""
import math

import torch

from shardcompute_amd.communicator import IdentityCommunicator
from shardcompute_amd.executor import DecodeGraph
from shardcompute_amd.kv_cache import KVCache
from shardcompute_amd.parallel.attention import ParallelAttention
from shardcompute_amd.parallel.mlp import ParallelMLP
from shardcompute_amd.parallel.quantized_linear import QuantizedColumnParallelLinear, QuantizedRowParallelLinear
from shardcompute_amd.parallel.transformer import ParallelTransformer, run_sync

GROUP = 64
EPS = 1e-5

# hidden, intermediate, q heads, kv heads, head_dim, vocab of one rank's share
SHAPES = {
    "tinyllama": dict(hidden=2048, inter=5632, heads=32, kv=4, dim=64, vocab=32000, theta=10000.0),
    "llama3-8b": dict(hidden=4096, inter=14336, heads=32, kv=8, dim=128, vocab=128256, theta=500000.0),
    # rank 0 of 8: one kv head and its 8 q heads, an eighth of the intermediate and vocab rows
    "llama3-70b/8": dict(hidden=8192, inter=3584, heads=8, kv=1, dim=128, vocab=16032, theta=500000.0),
}


def listed():
    return [
        # the smallest call: one token through TinyLlama's o projection (launch and host latency)
        dict(name="o_tinyllama_w4_m1", kind="linear", row=True, bits=4, m=1, k=2048, n=2048, bias=False),
        # one token's logits: the widest batch-1 product, the lm_head of every decode step
        dict(name="lm_head_8b_w4_m1", kind="linear", row=False, bits=4, m=1, k=4096, n=128256, bias=False),
        # the down projection of a batch-16 decode step
        dict(name="down_8b_w4_m16", kind="linear", row=True, bits=4, m=16, k=14336, n=4096, bias=False),
        # a ragged batch of 45 sequences through the 70B shard's gate|up width, 8 bits, with a linear bias
        dict(name="gate_up_70b_w8_m45", kind="linear", row=False, bits=8, m=45, k=8192, n=7168, bias=True),
        # a short odd prompt through TinyLlama's MLP at 8 bits
        dict(name="mlp_tinyllama_w8_333", kind="mlp", shape="tinyllama", bits=8, tokens=333),
        # the headline prompt's MLP
        dict(name="mlp_8b_w4_2048", kind="mlp", shape="llama3-8b", bits=4, tokens=2048),
        # the largest prefill: 32 prompts of 1024 tokens on the 70B shard
        dict(name="mlp_70b_w8_32768", kind="mlp", shape="llama3-70b/8", bits=8, tokens=32768),
        # the headline prompt's attention layer (q|k|v, rotation and cache append, attention, o)
        dict(name="attn_prefill_8b_w4_2048", kind="attn_prefill", shape="llama3-8b", bits=4, batch=1, seq=2048, past=0),
        # three odd prompts through TinyLlama's attention (head_dim 64, 8 q heads per kv head)
        dict(name="attn_prefill_tinyllama_w4_3x701", kind="attn_prefill", shape="tinyllama", bits=4, batch=3, seq=701,
             past=0),
        # one decode step's attention layer for 16 sequences of 2048 positions
        dict(name="attn_decode_8b_w4_b16", kind="attn_decode", shape="llama3-8b", bits=4, batch=16, past=2047),
        # whole call: a 2048-token prompt through a four-layer cut of the 8B decoder to the last logits
        dict(name="prefill_8b_w4_4l_2048", kind="prefill", shape="llama3-8b", bits=4, layers=4, batch=1, seq=2048),
        # whole call: one greedy decode step of the full 8B decoder after 2048 positions
        dict(name="decode_8b_w4_32l", kind="decode", shape="llama3-8b", bits=4, layers=32, past=2048),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "mlp", "attn_prefill", "attn_prefill", "attn_decode", "prefill", "decode"])
    bits = rng.choice([4, 4, 8])
    shape = rng.choice(sorted(SHAPES))
    if kind == "linear":
        k = GROUP * _log_int(rng, 16, 224)
        if rng.random() < 0.7:
            k = max(1024, k // 512 * 512)          # the widths of real projections
        n = _log_int(rng, 256, 32768)
        if rng.random() < 0.7:
            n = n // 64 * 64
        m = _log_int(rng, 1, 4096)
        return dict(kind=kind, row=rng.random() < 0.5, bits=bits, m=m, k=k, n=n, bias=rng.random() < 0.3)
    if kind == "mlp":
        return dict(kind=kind, shape=shape, bits=bits, tokens=_log_int(rng, 1, 8192))
    if kind == "attn_prefill":
        seq = _log_int(rng, 9, 3000)
        batch = rng.randint(1, max(1, min(16, 8192 // seq)))
        past = rng.choice([0, 0, _log_int(rng, 1, 1500)])
        return dict(kind=kind, shape=shape, bits=bits, batch=batch, seq=seq, past=past)
    if kind == "attn_decode":
        return dict(kind=kind, shape=shape, bits=bits, batch=_log_int(rng, 1, 48), past=_log_int(rng, 16, 4000))
    if kind == "prefill":
        seq = _log_int(rng, 9, 2500)
        return dict(kind=kind, shape=shape, bits=bits, layers=rng.randint(2, 4),
                    batch=rng.randint(1, max(1, min(8, 2600 // seq))), seq=seq)
    return dict(kind=kind, shape=rng.choice(["tinyllama", "llama3-8b"]), bits=bits, layers=rng.randint(2, 12),
                past=_log_int(rng, 16, 2500))


# ---------------------------------------------------------------- inputs


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _bf16(g, *shape, scale=1.0):
    return torch.randn(shape, generator=g, device="cuda").mul_(scale).to(torch.bfloat16)


def _quantized(g, n, k, bits):
    """(packed codes int32 [n, k bits/32], scales, biases bf16 [n, k/64]) of an N(0, 0.02) weight."""
    top, per = 2 ** bits - 1, 32 // bits
    shifts = torch.arange(per, device="cuda", dtype=torch.int64) * bits
    out = []
    step = max(1, (1 << 25) // k)
    for r in range(0, n, step):
        rows = min(step, n - r)
        w = torch.randn((rows, k // GROUP, GROUP), generator=g, device="cuda").mul_(0.02)
        lo, hi = w.amin(-1), w.amax(-1)
        s, b = ((hi - lo) / top).to(torch.bfloat16), lo.to(torch.bfloat16)
        q = ((w - b.float()[..., None]) / s.float()[..., None]).round_().clamp_(0, top).to(torch.int64)
        word = (q.reshape(rows, k // per, per) << shifts).sum(-1)
        out.append((torch.where(word >= 2 ** 31, word - 2 ** 32, word).to(torch.int32), s, b))
    return tuple(torch.cat([p[i] for p in out]) for i in range(3))


def _dequant(w, bits, dtype=torch.float64):
    q, s, b = w
    per = 32 // bits
    shifts = torch.arange(per, device=q.device, dtype=torch.int32) * bits
    codes = ((q[..., None] >> shifts) & (2 ** bits - 1)).reshape(s.shape[0], s.shape[1], GROUP).to(dtype)
    return (codes * s.to(dtype)[..., None] + b.to(dtype)[..., None]).reshape(s.shape[0], -1)


def _attn_weights(g, c, bits):
    nq, nkv = c["heads"] * c["dim"], c["kv"] * c["dim"]
    return dict(q=_quantized(g, nq, c["hidden"], bits), k=_quantized(g, nkv, c["hidden"], bits),
                v=_quantized(g, nkv, c["hidden"], bits), o=_quantized(g, c["hidden"], nq, bits))


def _mlp_weights(g, c, bits):
    return dict(gate=_quantized(g, c["inter"], c["hidden"], bits), up=_quantized(g, c["inter"], c["hidden"], bits),
                down=_quantized(g, c["hidden"], c["inter"], bits))


def _norm_weight(g, hidden):
    return (1.0 + 0.1 * torch.randn(hidden, generator=g, device="cuda")).to(torch.bfloat16)


def _model_weights(g, c, bits, layers):
    out = dict(layers=[])
    for _ in range(layers):
        out["layers"].append(dict(ln1=_norm_weight(g, c["hidden"]), ln2=_norm_weight(g, c["hidden"]),
                                  attn=_attn_weights(g, c, bits), mlp=_mlp_weights(g, c, bits)))
    out["embed"] = _bf16(g, c["vocab"], c["hidden"], scale=0.02)
    out["norm"] = _norm_weight(g, c["hidden"])
    out["head"] = _quantized(g, c["vocab"], c["hidden"], bits)
    return out


def _capacity(case):
    return (case.get("past", 0) + case.get("seq", 1) + 31) // 32 * 32


def _past(g, case, c, batch, layers):
    """Cached positions: rotated keys and values [batch, kv heads, past, dim] of each layer."""
    shape = (batch, c["kv"], case.get("past", 0), c["dim"])
    return [(_bf16(g, *shape), _bf16(g, *shape)) for _ in range(layers)]


def _inputs(case, seed):
    g, kind = _gen(seed), case["kind"]
    c = SHAPES[case["shape"]] if "shape" in case else None
    if kind == "linear":
        return dict(w=_quantized(g, case["n"], case["k"], case["bits"]), x=_bf16(g, case["m"], case["k"]),
                    bias=_bf16(g, case["n"]) if case["bias"] else None)
    if kind == "mlp":
        return dict(w=_mlp_weights(g, c, case["bits"]), x=_bf16(g, 1, case["tokens"], c["hidden"]))
    if kind in ("attn_prefill", "attn_decode"):
        s = case.get("seq", 1)
        return dict(w=_attn_weights(g, c, case["bits"]), x=_bf16(g, case["batch"], s, c["hidden"]),
                    past=_past(g, case, c, case["batch"], 1))
    b, s = case.get("batch", 1), case.get("seq", 1)
    return dict(w=_model_weights(g, c, case["bits"], case["layers"]),
                ids=torch.randint(0, c["vocab"], (b, s), generator=g, device="cuda"),
                past=_past(g, case, c, b, case["layers"]))


# ---------------------------------------------------------------- the program


def _load_attention(att, w):
    att.load_quantized_shards(*w["q"], None, *w["k"], None, *w["v"], None, *w["o"], None)
    att.qkv.build()


def _load_mlp(mlp, w):
    mlp.load_quantized_shards(*w["up"], None, *w["down"], None, *w["gate"], None)
    mlp.gate_up.build()


def _attention(c, case):
    return ParallelAttention(c["hidden"], c["heads"], 1, 0, num_kv_heads=c["kv"], head_dim=c["dim"],
                             max_position_embeddings=_capacity(case), rope_base=c["theta"], use_quantized=True,
                             quantization_bits=case["bits"])


def _model(c, case, w):
    # a rank's share of a wider model keeps the wider model's head count: rank 0 of 8
    ws = 8 if c["hidden"] // c["dim"] != c["heads"] else 1
    m = ParallelTransformer(vocab_size=c["vocab"] * ws, hidden_size=c["hidden"], num_layers=case["layers"],
                            num_heads=c["heads"] * ws, intermediate_size=c["inter"] * ws, world_size=ws, rank=0,
                            communicator=IdentityCommunicator(0, ws), num_kv_heads=c["kv"] * ws,
                            max_position_embeddings=_capacity(case), rms_norm_eps=EPS, rope_base=c["theta"],
                            use_quantized=True, quantization_bits=case["bits"], embedding="vocab",
                            quantized_lm_head=True)
    for layer, lw in zip(m.layers, w["layers"]):
        layer.input_layernorm.load_weights(lw["ln1"])
        layer.post_attention_layernorm.load_weights(lw["ln2"])
        _load_attention(layer.attention, lw["attn"])
        _load_mlp(layer.mlp, lw["mlp"])
        layer.attention.rope.tables(_capacity(case), m.device)
    m.load_embedding_weights(w["embed"])
    m.load_norm_weights(w["norm"])
    m.load_quantized_lm_head_weights(*w["head"])
    return m


def prepare(case, seed):
    kind, inp = case["kind"], _inputs(case, seed)
    if kind == "linear":
        cls = QuantizedRowParallelLinear if case["row"] else QuantizedColumnParallelLinear
        lin = cls(case["k"], case["n"], 1, 0, bias=case["bias"], bits=case["bits"])
        lin.load_quantized_shard(*inp["w"], inp["bias"])
        return dict(kind=kind, layer=lin, x=inp["x"])
    c = SHAPES[case["shape"]]
    if kind == "mlp":
        mlp = ParallelMLP(c["hidden"], c["inter"], 1, 0, use_quantized=True, quantization_bits=case["bits"])
        _load_mlp(mlp, inp["w"])
        return dict(kind=kind, layer=mlp, x=inp["x"])
    if kind in ("attn_prefill", "attn_decode"):
        att = _attention(c, case)
        _load_attention(att, inp["w"])
        att.rope.tables(_capacity(case), torch.device("cuda"))
        cache = KVCache(1, case["batch"], c["kv"], c["dim"], _capacity(case))
        cache.load_tuples(inp["past"])
        return dict(kind=kind, layer=att, x=inp["x"], cache=cache)
    model = _model(c, case, inp["w"])
    if kind == "prefill":
        cache = model.new_cache(case["batch"], _capacity(case))
        return dict(kind=kind, layer=model, ids=inp["ids"], cache=cache)
    cache = model.new_cache(1, _capacity(case))
    cache.load_tuples(inp["past"])
    # decode as generate() sets it up: the step's buffers, plan and graph are kept
    dec = DecodeGraph(model, cache, torch.zeros((1, 1), dtype=torch.int32, device="cuda"))
    st = dict(kind=kind, layer=dec, ids=inp["ids"].to(torch.int32), cache=cache, counters=cache.counters.clone(),
              past=case["past"])
    run(st)
    return st


def run(state):
    kind, layer = state["kind"], state["layer"]
    if kind == "linear" or kind == "mlp":
        return run_sync(layer.forward(state["x"]))
    cache = state["cache"]
    if kind in ("attn_prefill", "attn_decode"):
        # the layer appends at the cache's length, which the model advances after its
        # last layer: a further pass appends the same positions again
        out, kv = run_sync(layer.forward(state["x"], past_key_value=cache[0], use_cache=True))
        return out, kv.k, kv.vt
    if kind == "prefill":
        cache.reset()
        logits, kv = run_sync(layer.forward(state["ids"], past_key_values=cache, use_cache=True, last_only=True))
        return logits, kv.k, kv.vt
    # one decode step of the given token at the given position
    cache.length = state["past"]
    cache.counters.copy_(state["counters"])
    layer.bufs.ids.copy_(state["ids"])
    layer.run(1)
    return layer.logits, cache.k, cache.vt


# ---------------------------------------------------------------- work and accuracy


def _mat_bytes(n, k, bits):
    return n * k * bits // 8 + n * (k // GROUP) * 4


def _attn_core(c, b, s, past):
    """(bytes, flops) of the attention itself: q, k, v in, k and v appended, the cached positions read, output."""
    nq, nkv = c["heads"] * c["dim"], c["kv"] * c["dim"]
    nbytes = 2 * b * (2 * nkv * past + s * 2 * nkv)
    return nbytes, 4 * b * nq * (s * past + s * (s + 1) // 2)


def _proj(c, bits, names):
    nq, nkv, h, i = c["heads"] * c["dim"], c["kv"] * c["dim"], c["hidden"], c["inter"]
    dims = dict(q=(nq, h), k=(nkv, h), v=(nkv, h), o=(h, nq), gate=(i, h), up=(i, h), down=(h, i))
    return (sum(_mat_bytes(*dims[p], bits) for p in names), sum(2 * dims[p][0] * dims[p][1] for p in names))


def work(case):
    kind, bits = case["kind"], case["bits"]
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return dict(bytes=_mat_bytes(n, k, bits) + 2 * m * (k + n) + (2 * n if case["bias"] else 0),
                    flops=2 * m * n * k)
    c = SHAPES[case["shape"]]
    if kind == "mlp":
        wb, wf = _proj(c, bits, ("gate", "up", "down"))
        return dict(bytes=wb + 4 * case["tokens"] * c["hidden"], flops=case["tokens"] * wf)
    b, s, past = case.get("batch", 1), case.get("seq", 1), case.get("past", 0)
    ab, af = _attn_core(c, b, s, past)
    if kind in ("attn_prefill", "attn_decode"):
        wb, wf = _proj(c, bits, ("q", "k", "v", "o"))
        return dict(bytes=wb + ab + 4 * b * s * c["hidden"], flops=b * s * wf + af)
    wb, wf = _proj(c, bits, ("q", "k", "v", "o", "gate", "up", "down"))
    return dict(bytes=case["layers"] * (wb + ab) + 2 * b * s * c["hidden"] + _mat_bytes(c["vocab"], c["hidden"], bits)
                + 2 * b * c["vocab"],
                flops=case["layers"] * (b * s * wf + af) + 2 * b * c["vocab"] * c["hidden"])


def tolerance(case):
    """About four times the 2-norm error of this path against ``exact`` (bf16 activations and
    weights dequantized to bf16: 0.0017-0.0035 a product, 0.0045 the MLP's two, 0.0067 the
    attention layer's projections and probabilities; 0.014-0.023 the logits of 2-4 layers
    and 0.046 of 32, a rounding in one layer travelling through all that follow)."""
    kind = case["kind"]
    if kind in ("prefill", "decode"):
        return {"rel": 0.08 + 0.003 * case["layers"]}
    return {"rel": {"linear": 0.012, "mlp": 0.018}.get(kind, 0.025)}


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _rotate(x, pos, theta):
    """x [..., positions, dim] rotated (half-split pairs) for the given positions."""
    d = x.shape[-1]
    ang = pos.double()[:, None] * (theta ** (-torch.arange(0, d, 2, device=x.device).double() / d))
    cs, sn = torch.cos(ang), torch.sin(ang)
    a, b = x[..., :d // 2], x[..., d // 2:]
    return torch.cat([a * cs - b * sn, b * cs + a * sn], -1)


def _exact_attention(x, w, past, c, bits, theta):
    """x [b, s, hidden] -> (output, keys, values), keys and values [b, kv, past + s, dim]."""
    b, s, _ = x.shape
    h, kv, d, t0 = c["heads"], c["kv"], c["dim"], past[0].shape[2]
    pos = torch.arange(t0, t0 + s, device=x.device)
    q = (x @ _dequant(w["q"], bits).T).view(b, s, h, d).transpose(1, 2)
    k = (x @ _dequant(w["k"], bits).T).view(b, s, kv, d).transpose(1, 2)
    v = (x @ _dequant(w["v"], bits).T).view(b, s, kv, d).transpose(1, 2)
    q = _rotate(q, pos, theta)
    k = torch.cat([past[0].double(), _rotate(k, pos, theta)], 2)
    v = torch.cat([past[1].double(), v], 2)
    out = torch.empty((b, s, h * d), dtype=torch.float64, device=x.device)
    hidden_keys = torch.arange(t0 + s, device=x.device)[None, :] > pos[:, None]
    for i in range(b):
        for j in range(h):
            sc = (q[i, j] @ k[i, j * kv // h].T) / math.sqrt(d)
            p = torch.softmax(sc.masked_fill_(hidden_keys, -math.inf), -1)
            out[i, :, j * d:(j + 1) * d] = p @ v[i, j * kv // h]
    return out @ _dequant(w["o"], bits).T, k, v


def _exact_mlp(x, w, bits):
    out = torch.empty_like(x)
    gate, up, down = (_dequant(w[p], bits).T for p in ("gate", "up", "down"))
    for r in range(0, x.shape[0], 8192):
        g = x[r:r + 8192] @ gate
        out[r:r + 8192] = (g * torch.sigmoid(g) * (x[r:r + 8192] @ up)) @ down
    return out


def _cache_layout(k, v, cap):
    """keys [b, kv, t, d] and values in the cache's buffers [b, kv, cap, d] and [b, kv, d, cap]."""
    pad = cap - k.shape[2]
    kc = torch.nn.functional.pad(k, (0, 0, 0, pad))
    return kc, torch.nn.functional.pad(v, (0, 0, 0, pad)).transpose(2, 3)


def exact(case, seed):
    kind, bits, inp = case["kind"], case["bits"], _inputs(case, seed)
    if kind == "linear":
        out = inp["x"].double() @ _dequant(inp["w"], bits).T
        return out + inp["bias"].double() if case["bias"] else out
    c = SHAPES[case["shape"]]
    if kind == "mlp":
        return _exact_mlp(inp["x"][0].double(), inp["w"], bits)[None]
    cap = _capacity(case)
    if kind in ("attn_prefill", "attn_decode"):
        out, k, v = _exact_attention(inp["x"].double(), inp["w"], inp["past"][0], c, bits, c["theta"])
        return (out, *_cache_layout(k, v, cap))
    w, h = inp["w"], inp["w"]["embed"][inp["ids"]].double()
    ks, vs = [], []
    for lw, past in zip(w["layers"], inp["past"]):
        a, k, v = _exact_attention(_rms(h, lw["ln1"]), lw["attn"], past, c, bits, c["theta"])
        h = h + a
        xn = _rms(h, lw["ln2"])
        h = h + _exact_mlp(xn.reshape(-1, c["hidden"]), lw["mlp"], bits).view(h.shape)
        kc, vt = _cache_layout(k, v, cap)
        ks.append(kc)
        vs.append(vt)
    logits = _rms(h[:, -1:], w["norm"]) @ _dequant(w["head"], bits).T
    if kind == "decode":
        logits = logits[:, 0]
    return logits, torch.stack(ks), torch.stack(vs)
