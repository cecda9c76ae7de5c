"""Performance cases of the framework: what its users have it do, through its public entry points.

The kinds of cases, and the entry point each one times:

* ``gemv``    the decode product, ``torch.ops.binary_kernels.nanoquant_dyn_forward``;
* ``gemm``    the prefill product, ``torch.ops.binary_kernels.marlin_nanoquant_forward``;
* ``linear``  a ``NanoQuantLinear`` prepared for ``auto``, called as a module on a 3-D input;
* ``pack``    dense +-1 factors to the words of both kernels (what preparing a layer does);
* ``words``   checkpoint words to the words of both kernels (what loading a packed layer does);
* ``layer``   one decoder layer over a whole prompt, or over a chunk after a cached context;
* ``prompt``  ``FusedDecoder.prefill``: a whole prompt through a small model, logits at its end;
* ``decode``  ``FusedDecoder.decode``: one graph-replayed token step of a small model.

The linear shapes are those of ``bench.py`` (Llama-2-7B and Llama-3-70B at 0.55 bits per weight);
models keep a few of their layers. Weights, scales and activations are drawn from the seed: signs
are fair coins, scales |N(1, 0.2)| over the root of the summed length (so that a unit-RMS input
gives a unit-RMS output), activations N(0, 1), token ids uniform.
"""
import math

import torch
import torch.nn as nn

import nanoquant_amd  # noqa: F401  registers torch.ops.binary_kernels.*
from nanoquant_amd.decode import FusedDecoder, LlamaShape, NanoQuantLlama, StaticKVCache
from nanoquant_amd.kernel import utils as packers
from nanoquant_amd.modules.linear import NanoQuantLinear

DEVICE = "cuda"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
EPS, THETA = 1e-5, 10000.0


# ------------------------------------------------------------------------------------- the cases

def listed():
    return [
        # one token through an attention projection of a 7B layer: the smallest call there is
        dict(name="gemv_q_1", kind="gemv", m=4096, n=4096, r=1120, rows=1, dtype="fp16", mid=False),
        # four sequences through a 70B gate projection: a tall layer, bf16, with its middle scale
        dict(name="gemv_gate70_4", kind="gemv", m=28672, n=8192, r=3520, rows=4, dtype="bf16", mid=True),
        # a prompt of 300 tokens through a 7B gate projection packed for decoding only
        dict(name="gemv_gate_300", kind="gemv", m=11008, n=4096, r=1632, rows=300, dtype="fp16", mid=False),
        # three sequences of seven tokens (a short continuation) through a 7B down projection
        dict(name="linear_down_21", kind="linear", m=4096, n=11008, r=1632, rows=7, batch=3, dtype="fp16", mid=True),
        # a long prompt through a 7B gate projection
        dict(name="gemm_gate_2048", kind="gemm", m=11008, n=4096, r=1632, rows=2048, dtype="fp16", mid=False),
        # a ragged batch of prompts through a 70B down projection: long sums, bf16
        dict(name="gemm_down70_333", kind="gemm", m=8192, n=28672, r=3520, rows=333, dtype="bf16", mid=True),
        # preparing a 7B down projection from its dense factors, and loading a 70B gate from a checkpoint's words
        dict(name="pack_down", kind="pack", m=4096, n=11008, r=1632, dtype="fp16"),
        dict(name="words_gate70", kind="words", m=28672, n=8192, r=3520, dtype="fp16"),
        # a 2048-token prompt through a 7B decoder layer
        dict(name="layer_2048", kind="layer", heads=32, kv_heads=32, ffn=11008, tokens=2048, past=0, batch=1,
             kernel="gemm", dtype="fp16"),
        # two ragged prompts through two grouped-query layers and the head (70B shapes)
        dict(name="prompt_gqa_333", kind="prompt", heads=64, kv_heads=8, ffn=28672, layers=2, tokens=333, batch=2,
             dtype="bf16", attention="hip"),
        # a chat's next token: one sequence, a 1000-token context, 7B layers, the default step
        dict(name="decode_1", kind="decode", heads=32, kv_heads=32, ffn=11008, layers=4, past=1000, batch=1,
             dtype="fp16", attention="torch"),
        # the next token of 16 sequences on grouped-query layers (70B shapes)
        dict(name="decode_gqa_16", kind="decode", heads=64, kv_heads=8, ffn=28672, layers=2, past=500, batch=16,
             dtype="bf16", attention="hip"),
    ]


def _spread(rng, low, high, step=1):
    """A multiple of ``step`` between the two, spread over its logarithm."""
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return max(step, int(round(v / step)) * step)


def _rank(rng, m, n):
    """The rank of 0.4 to 1 bits per weight, a multiple of 32 as the quantizer rounds it."""
    return max(32, int(round(rng.uniform(0.4, 1.0) * m * n / (m + n) / 32)) * 32)


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "gemm", "linear", "pack", "words", "layer", "prompt", "decode"])
    c = dict(kind=kind, dtype=rng.choice(["fp16", "bf16"]))
    if kind in ("gemv", "gemm", "linear", "pack", "words"):
        # the packers of the prefill product need m % 64 == 0 and n % 16 == 0; the decode product takes any
        # m and any n, 8 being the step of real hidden sizes
        ragged = kind == "gemv"
        m = _spread(rng, 1024, 28672, 1 if ragged else 64)
        n = _spread(rng, 1024, 28672, 8 if ragged else 64)
        if max(m, n) > 12288:  # real layers are wide or tall, not both
            m, n = (m, min(n, 8192)) if m > n else (min(m, 8192), n)
        c.update(m=m, n=n, r=_rank(rng, m, n))
    if kind in ("gemv", "gemm", "linear"):
        most = max(1, int(2.5e11 // (c["r"] * (m + n))))  # no costlier than the listed ones
        rows = _spread(rng, 16, 2048) if kind == "gemm" else _spread(rng, 1, 512)
        c.update(rows=max(1, min(rows, most)), mid=rng.random() < 0.5)
    if kind == "linear":
        c.update(batch=rng.choice([1, 2, 3]))
        c["rows"] = max(1, c["rows"] // c["batch"])
    if kind in ("layer", "prompt", "decode"):
        heads = rng.choice([8, 16, 24, 32])
        c.update(heads=heads, kv_heads=heads // rng.choice([1, 1, 4, 8]), ffn=_spread(rng, 256 * heads, 448 * heads, 64))
    if kind == "layer":
        c.update(batch=rng.choice([1, 1, 2]), kernel=rng.choice(["gemm", "auto"]), past=rng.choice([0, rng.randrange(1, 1000)]))
        c["tokens"] = _spread(rng, 64, 2000) // c["batch"]
    if kind == "prompt":
        c.update(batch=rng.choice([1, 2, 4]), layers=2, attention=rng.choice(["torch", "hip"]))
        c["tokens"] = _spread(rng, 64, 900) // c["batch"]
    if kind == "decode":
        c.update(batch=_spread(rng, 1, 32), layers=2, attention=rng.choice(["torch", "hip"]))
        c["past"] = min(_spread(rng, 64, 2000), 8000 // c["batch"])
    return c


# ------------------------------------------------------------------------------ inputs from a seed

def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _factors(g, m, n, r, dtype, mid):
    """One linear's factors: V [r, n] and U [m, r] as int8 signs, its scales in ``dtype``."""
    def signs(rows, cols):
        return torch.randint(0, 2, (rows, cols), dtype=torch.int8, device=DEVICE, generator=g).mul_(2).sub_(1)

    def scales(k, over):
        return ((torch.randn(k, device=DEVICE, generator=g) * 0.2 + 1.0).abs() / math.sqrt(over)).to(dtype)

    return {"V": signs(r, n), "U": signs(m, r), "pre": scales(n, n), "post": scales(m, r),
            "mid": scales(r, 1.0) if mid else None}


def _normal(g, shape, dtype):
    return torch.randn(shape, device=DEVICE, generator=g).to(dtype)


def _shape(case):
    hidden = 128 * case["heads"]
    return LlamaShape(hidden=hidden, layers=case.get("layers", 1), heads=case["heads"], kv_heads=case["kv_heads"],
                      ffn=case["ffn"], vocab=32000, rms_eps=EPS, rope_theta=THETA)


def _bpw_rank(m, n):
    return max(32, int(round(0.55 * m * n / (m + n) / 32)) * 32)


def _layer_factors(case, g):
    """Name -> factors of a decoder layer's seven linears, and its two norm weights."""
    h, kv, f = 128 * case["heads"], 128 * case["kv_heads"], case["ffn"]
    dt = DTYPES[case["dtype"]]
    sizes = {"q_proj": (h, h), "k_proj": (kv, h), "v_proj": (kv, h), "o_proj": (h, h), "gate_proj": (f, h),
             "up_proj": (f, h), "down_proj": (h, f)}
    out = {name: _factors(g, m, n, _bpw_rank(m, n), dt, False) for name, (m, n) in sizes.items()}
    for name in ("input_layernorm", "post_attention_layernorm"):
        out[name] = (torch.randn(h, device=DEVICE, generator=g) * 0.1 + 1.0).to(dt)
    return out


def _model_weights(case, g):
    dt, h = DTYPES[case["dtype"]], 128 * case["heads"]
    return {"embed": _normal(g, (32000, h), dt), "head": (_normal(g, (32000, h), dt) / math.sqrt(h)).to(dt),
            "norm": (torch.randn(h, device=DEVICE, generator=g) * 0.1 + 1.0).to(dt),
            "layers": [_layer_factors(case, g) for _ in range(case["layers"])]}


# -------------------------------------------------------------------------------- what a user keeps

def _linear(f, kernel, dtype):
    m, n, r = f["U"].shape[0], f["V"].shape[1], f["V"].shape[0]
    lin = nn.Linear(n, m, device="meta")
    lin.bias = nn.Parameter(torch.zeros(m, device=DEVICE), requires_grad=False)  # the device of the new parameters
    lin.__class__ = NanoQuantLinear
    lin.init_for_inference(r, has_scale_mid=f["mid"] is not None)
    lin.bias = None
    for name, value in (("V", f["V"]), ("U", f["U"])):
        getattr(lin, name).data = value.to(torch.bfloat16)
    # the scales as given: init_for_inference's are bf16, too coarse for a float16 layer
    for name, key in (("scale_pre", "pre"), ("scale_post", "post"), ("scale_mid", "mid")):
        if f[key] is not None:
            getattr(lin, name).data = f[key].view(1, -1)
    lin._prepare_kernel(kernel, dtype)
    return lin


def _fill_layer(layer, w, kernel, dtype):
    for name in ("q_proj", "k_proj", "v_proj", "o_proj"):
        setattr(layer.self_attn, name, _linear(w[name], kernel, dtype))
    for name in ("gate_proj", "up_proj", "down_proj"):
        setattr(layer.mlp, name, _linear(w[name], kernel, dtype))
    for name in ("input_layernorm", "post_attention_layernorm"):
        getattr(layer, name).weight.data.copy_(w[name])


def _model(case, w):
    dt = DTYPES[case["dtype"]]
    model = NanoQuantLlama(_shape(case), device=DEVICE, dtype=dt)
    model.model.embed_tokens.weight.data.copy_(w["embed"])
    model.lm_head.weight.data.copy_(w["head"])
    model.model.norm.weight.data.copy_(w["norm"])
    for layer, lw in zip(model.model.layers, w["layers"]):
        _fill_layer(layer, lw, "gemv", dt)
    return model.cast_non_linears(dt).eval()


def _tokens(case, g, count):
    return torch.randint(0, 32000, (case["batch"], count), device=DEVICE, generator=g)


def _inputs(case, seed):
    """Everything drawn for a case: weights, and the activations or tokens."""
    g, kind, dt = _generator(seed), case["kind"], DTYPES[case["dtype"]]
    if kind in ("gemv", "gemm", "linear", "pack", "words"):
        f = _factors(g, case["m"], case["n"], case["r"], dt, case.get("mid", kind in ("pack", "words")))
        lead = (case["batch"], case["rows"]) if kind == "linear" else (case.get("rows", 1),)
        return f, _normal(g, lead + (case["n"],), dt)
    if kind == "layer":
        kv = (case["batch"], case["kv_heads"], case["past"], 128)
        return _layer_factors(case, g), (_normal(g, (case["batch"], case["tokens"], 128 * case["heads"]), dt),
                                         _normal(g, kv, dt), _normal(g, kv, dt))
    return _model_weights(case, g), _tokens(case, g, case["tokens"] if kind == "prompt" else case["past"] + 1)


def prepare(case, seed):
    kind, dt = case["kind"], DTYPES[case["dtype"]]
    w, x = _inputs(case, seed)
    if kind == "gemv":
        return kind, (x, w["pre"], packers.binary_packer(w["V"], "half2"), w["mid"],
                      packers.binary_packer(w["U"], "half2"), w["post"])
    if kind == "gemm":
        mid = w["mid"] if w["mid"] is not None else torch.ones(case["r"], device=DEVICE, dtype=dt)
        words_v, words_u, pre, mid, post, ws = packers.marlin_nanoquant_packer(w["V"].T, w["U"].T, w["pre"], mid, w["post"])
        return kind, (x, words_v, words_u, pre, mid, post, ws)
    if kind == "linear":
        return kind, (_linear(w, "auto", dt), x)
    if kind == "pack":
        return kind, w
    if kind == "words":
        return kind, dict(w, V=packers.binary_packer(w["V"]), U=packers.binary_packer(w["U"]), m=case["m"], n=case["n"],
                          r=case["r"])
    if kind == "layer":
        s, past, x, k, v = _shape(case), case["past"], *x
        model = NanoQuantLlama(LlamaShape(**dict(vars(s), vocab=64)), device=DEVICE, dtype=dt)
        layer = model.model.layers[0]
        _fill_layer(layer, w, case["kernel"], dt)
        cache = StaticKVCache(s, case["batch"], past + case["tokens"] + 64, DEVICE, dt)
        cache.k[0][:, :, :past].copy_(k)
        cache.v[0][:, :, :past].copy_(v)
        positions = torch.arange(past, past + case["tokens"], device=DEVICE)
        cos, sin = model.rope(positions, dt)
        return kind, (layer, x, cos, sin, positions, cache)
    past = case["tokens"] if kind == "prompt" else case["past"]
    decoder = FusedDecoder(_model(case, w), case["batch"], past + 256, attention=case["attention"])
    if kind == "prompt":
        return kind, (decoder, x)
    decoder.capture()
    decoder.prefill(x[:, :past])
    return kind, (decoder, past, x[:, past].clone())


# -------------------------------------------------------------------------------------------- a pass

def run(state):
    kind, s = state
    with torch.no_grad():
        if kind == "gemv":
            return torch.ops.binary_kernels.nanoquant_dyn_forward(*s, 128, 128, 2, 2, 1, 1, 8, 8)
        if kind == "gemm":
            return torch.ops.binary_kernels.marlin_nanoquant_forward(*s)
        if kind == "linear":
            return s[0](s[1])
        if kind == "pack":
            return [packers.binary_packer(s["V"], "half2"), packers.binary_packer(s["U"], "half2"),
                    *packers.marlin_nanoquant_packer(s["V"].T, s["U"].T, s["pre"], s["mid"], s["post"])]
        if kind == "words":
            sizes = ((s["r"], s["n"]), (s["m"], s["r"]))
            return [packers.repack_binary_gemv(s["V"], sizes[0], "lsb_first", "half2"),
                    packers.repack_binary_gemv(s["U"], sizes[1], "lsb_first", "half2"),
                    *packers.pack_binary_marlin_fused_from_packed(s["V"], sizes[0], s["U"], sizes[1], s["pre"], s["mid"],
                                                                  s["post"])]
        if kind == "layer":
            layer, x, cos, sin, positions, cache = s
            return layer(x, cos, sin, positions, cache), cache.k[0], cache.v[0]
        if kind == "prompt":
            decoder, ids = s
            logits = decoder.prefill(ids)
            return [logits, *decoder.cache.v]
        decoder, past, token = s  # the step of the token after the context, as a program scoring a reply runs it
        decoder.pos.fill_(past)
        decoder.tok.copy_(token)
        return [decoder.decode(1), *decoder.cache.v]


# --------------------------------------------------------------------- what a pass cannot do without

def _layer_linears(case):
    h, kv, f = 128 * case["heads"], 128 * case["kv_heads"], case["ffn"]
    return [(h, h), (kv, h), (kv, h), (h, h), (f, h), (f, h), (h, f)]


def _linear_bytes(m, n, r):
    return r * n / 8 + m * r / 8 + 2 * (m + n)


def work(case):
    kind = case["kind"]
    if kind in ("gemv", "gemm", "linear"):
        m, n, r, rows = case["m"], case["n"], case["r"], case["rows"] * case.get("batch", 1)
        return {"bytes": _linear_bytes(m, n, r) + 2 * rows * (m + n) + 2 * r * case["mid"],
                "flops": 2.0 * rows * r * (m + n)}
    if kind in ("pack", "words"):
        signs = case["r"] * (case["m"] + case["n"])
        return {"bytes": signs * (1.0 if kind == "pack" else 1 / 8) + 2 * signs / 8 + 4 * (case["m"] + case["n"]),
                "flops": 0}
    h, kv, batch, layers = 128 * case["heads"], 128 * case["kv_heads"], case["batch"], case.get("layers", 1)
    tokens = case.get("tokens", 1)
    past = case.get("past", 0)
    keys = tokens * past + tokens * (tokens + 1) / 2  # (query, key) pairs of a sequence and head
    per_layer = sum(2.0 * batch * tokens * _bpw_rank(m, n) * (m + n) for m, n in _layer_linears(case))
    per_layer += 4.0 * batch * keys * h
    nbytes = sum(_linear_bytes(m, n, _bpw_rank(m, n)) for m, n in _layer_linears(case))
    nbytes += 4 * batch * (past + tokens) * kv  # the context's keys and values read, the new ones written
    flops, nbytes = layers * per_layer, layers * nbytes
    if kind == "layer":
        return {"bytes": nbytes + 4 * batch * tokens * h, "flops": flops}
    return {"bytes": nbytes + 2 * 32000 * h + 4 * batch * 32000, "flops": flops + 2.0 * batch * h * 32000}


def tolerance(case):
    kind, half = case["kind"], case["dtype"] == "fp16"
    if kind in ("pack", "words"):
        return "exact"
    return {"rel": TOLERANCE[kind][0 if half else 1]}


# About four times the error that a run shows against `exact`. The outputs' own rounding is 2.1e-4 (fp16) and
# 1.7e-3 (bf16) of their 2-norm; the prefill product also rounds its intermediate, a layer a dozen tensors and a
# model all of its layers'.
TOLERANCE = {"gemv": (1e-3, 7e-3), "linear": (1.2e-3, 1e-2), "gemm": (1.2e-3, 1e-2), "layer": (2e-3, 1.6e-2),
             "prompt": (5e-3, 3e-2), "decode": (5e-3, 3e-2)}


# ----------------------------------------------------------------------------------- 64-bit reference

def _exact_linear(f, x):
    h = (x * f["pre"].double()) @ f["V"].double().T
    if f["mid"] is not None:
        h = h * f["mid"].double()
    return (h @ f["U"].double().T) * f["post"].double()


def _exact_norm(x, weight):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * weight.double()


def _exact_rope(x, positions, dt):
    """Rotate-half on [..., T, 128], with the tables in the dtype that the path is given them in."""
    inv = 1.0 / (THETA ** (torch.arange(0, 128, 2, dtype=torch.float32, device=x.device) / 128))
    a = positions.float().view(-1, 1) * inv
    cos, sin = (t(torch.cat((a, a), -1)).to(dt).double() for t in (torch.cos, torch.sin))
    return x * cos + torch.cat((-x[..., 64:], x[..., :64]), -1) * sin


def _exact_layer(case, w, x, k_past, v_past, positions):
    """Hidden states after a layer, with the keys and values of the whole context."""
    B, T, H, KV = x.shape[0], x.shape[1], case["heads"], case["kv_heads"]
    dt = DTYPES[case["dtype"]]
    a = _exact_norm(x, w["input_layernorm"])
    q, k, v = (_exact_linear(w[p], a).view(B, T, -1, 128).transpose(1, 2) for p in ("q_proj", "k_proj", "v_proj"))
    q, k = _exact_rope(q, positions, dt), _exact_rope(k, positions, dt)
    k, v = torch.cat((k_past.double(), k), 2), torch.cat((v_past.double(), v), 2)
    hidden = torch.arange(k.shape[2], device=x.device).view(1, -1) > positions.view(-1, 1)
    out = torch.empty_like(q)
    for b in range(B):
        for i in range(H):  # a head at a time: the scores of all would not fit
            s = (q[b, i] @ k[b, i * KV // H].T) * 128 ** -0.5
            out[b, i] = torch.softmax(s.masked_fill_(hidden, -math.inf), -1) @ v[b, i * KV // H]
    x = x + _exact_linear(w["o_proj"], out.transpose(1, 2).reshape(B, T, -1))
    a = _exact_norm(x, w["post_attention_layernorm"])
    gate, up = _exact_linear(w["gate_proj"], a), _exact_linear(w["up_proj"], a)
    return x + _exact_linear(w["down_proj"], nn.functional.silu(gate) * up), k, v


def exact(case, seed):
    kind = case["kind"]
    if kind in ("pack", "words"):
        return None  # whole numbers and moved scales: compared bit for bit
    w, x = _inputs(case, seed)
    if kind in ("gemv", "gemm", "linear"):
        return _exact_linear(w, x.double())
    if kind == "layer":
        x, k_past, v_past = x
        positions = torch.arange(case["past"], case["past"] + case["tokens"], device=DEVICE)
        y, k, v = _exact_layer(case, w, x.double(), k_past, v_past, positions)
        room = (0, 0, 0, 64)  # the cache's unused rows
        return y, nn.functional.pad(k, room), nn.functional.pad(v, room)
    ids, none = x, torch.empty(case["batch"], case["kv_heads"], 0, 128, device=DEVICE)
    positions = torch.arange(ids.shape[1], device=DEVICE)
    h, values = w["embed"][ids].double(), []
    for lw in w["layers"]:
        h, _, v = _exact_layer(case, lw, h, none, none, positions)
        values.append(v)
    logits = _exact_norm(h[:, -1], w["norm"]) @ w["head"].double().T
    room = (0, 0, 0, 255 if kind == "decode" else 256)  # the caches' unused rows
    return [logits, *(nn.functional.pad(v, room) for v in values)]
