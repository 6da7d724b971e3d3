"""The work a program has this framework do, as cases that can be timed and checked.

A case is a dict of plain values; `prepare` makes on the GPU what a program holds before the call
(tensors, weights, a model), `run` makes one pass through the framework's public entry points and
returns its whole outputs, `exact` gives the same outputs in float64 by plain torch.

Kinds (field "kind"), each a layer, a block or a whole call of a transformer:
  attention  scaled dot-product attention of a prompt (prefill), causal, grouped-query heads
  decode     one query token per sequence against KV caches of mixed lengths
  norm_rope  the hidden RMSNorm and the per-head qk-norm + RoPE of a chunk of tokens
  qkv        a chunk's QKV projection with qk-norm, RoPE and the KV-cache write
  mlp        RMSNorm, SwiGLU and the down projection with the residual add
  linear     one projection (y = x W^T + b)
  forward    a Qwen3 model's forward over a prompt: the logits of its last position
  generate   a Qwen3 model's prefill and greedy decoding: every step's logits and the tokens
"""
import math

import numpy as np
import torch

from kandle_amd import HipBackend, Tensor, env
from kandle_amd import functional as F
from kandle_amd.model_utils.qwen3 import Qwen3Config, Qwen3ForCausalLM, weight_names, weight_shape

EPS = 1e-6
THETA = 1e6
VOCAB = 151936
# hidden, intermediate, query heads, kv heads of the Qwen3 sizes this framework's tests run
WIDTHS = {"0.6b": (1024, 3072, 16, 8), "4b": (2560, 9728, 32, 8), "14b": (5120, 17408, 40, 8)}


def listed():
    return [
        # Batched long prompts on the bf16 path: four full 4096-token contexts.
        {"name": "attention_bf16_4x4096", "kind": "attention", "dtype": "bfloat16", "split": False, "batch": 4, "hq": 16,
         "hkv": 8, "s": 4096, "d": 128, "causal": True, "heads_first": True},
        # One user's prompt of an ordinary, odd length, read as [batch, seq, head, dim] views of the projections.
        {"name": "attention_bf16_1x1531", "kind": "attention", "dtype": "bfloat16", "split": False, "batch": 1, "hq": 16,
         "hkv": 8, "s": 1531, "d": 128, "causal": True, "heads_first": False},
        # The prompt attention of the float32-activation model, which is the default.
        {"name": "attention_f32_split_1x512", "kind": "attention", "dtype": "float32", "split": True, "batch": 1,
         "hq": 16, "hkv": 8, "s": 512, "d": 128, "causal": True, "heads_first": True},
        # The plain float32 attention call on a short prompt: latency and launches count.
        {"name": "attention_f32_1x256", "kind": "attention", "dtype": "float32", "split": False, "batch": 1, "hq": 16,
         "hkv": 8, "s": 256, "d": 128, "causal": True, "heads_first": True},
        # Serving eight long conversations: one token each over 8k to 32k cached keys.
        {"name": "decode_bf16_8x32768", "kind": "decode", "dtype": "bfloat16", "batch": 8, "hq": 16, "hkv": 8,
         "len": 32768, "d": 128},
        # Serving a few short chats from float32 caches: the smallest attention call.
        {"name": "decode_f32_2x777", "kind": "decode", "dtype": "float32", "batch": 2, "hq": 16, "hkv": 8, "len": 777,
         "d": 128},
        # Norms and rotary embedding of a long chunk (memory bound).
        {"name": "norm_rope_bf16_8192", "kind": "norm_rope", "dtype": "bfloat16", "tokens": 8192, "width": "0.6b"},
        # The attention input of a 512-token prompt, float32 activations over bf16 weights (the default).
        {"name": "qkv_f32_512", "kind": "qkv", "dtype": "float32", "tokens": 512, "width": "0.6b"},
        # The MLP block of the same prompt.
        {"name": "mlp_f32_512", "kind": "mlp", "dtype": "float32", "tokens": 512, "width": "0.6b"},
        # The MLP block of a larger model over a long bf16 chunk: where matrix throughput counts.
        {"name": "mlp_bf16_2000", "kind": "mlp", "dtype": "bfloat16", "tokens": 2000, "width": "4b"},
        # A whole prompt of an ordinary length through the model.
        {"name": "forward_f32_1000", "kind": "forward", "dtype": "float32", "tokens": 1000},
        # A whole answer: prompt, then token after token, the logits of each read by the program.
        {"name": "generate_f32_512_32", "kind": "generate", "dtype": "float32", "tokens": 512, "new": 32},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["attention", "attention", "attention", "decode", "decode", "norm_rope", "qkv", "mlp", "mlp",
                       "linear", "linear", "forward", "generate"])
    dtype = rng.choice(["bfloat16", "float32"])
    if kind == "attention":
        hq, hkv = rng.choice([(16, 8), (32, 8), (40, 8), (16, 16)])
        f32 = dtype == "float32"
        s = _log(rng, 64, 2048 if f32 else 4096)
        return {"kind": kind, "dtype": dtype, "split": f32 and rng.random() < 0.6, "batch": rng.choice([1, 1, 1, 2] if
                (f32 or hq > 16) else [1, 1, 2, 4]), "hq": hq, "hkv": hkv, "s": s, "d": rng.choice([128, 128, 128, 64]),
                "causal": rng.random() < 0.85, "heads_first": rng.random() < 0.5}
    if kind == "decode":
        hq, hkv = rng.choice([(16, 8), (32, 8), (40, 8), (16, 16)])
        batch = rng.randint(1, 8)
        most = 32768 if dtype == "bfloat16" and hkv == 8 else 16384
        return {"kind": kind, "dtype": dtype, "batch": batch, "hq": hq, "hkv": hkv, "len": _log(rng, 128, most),
                "d": rng.choice([128, 128, 64])}
    if kind == "norm_rope":
        return {"kind": kind, "dtype": dtype, "tokens": _log(rng, 32, 8192), "width": rng.choice(["0.6b", "4b"])}
    if kind in ("qkv", "mlp", "linear"):
        width = rng.choice(["0.6b", "0.6b", "4b", "14b"])
        case = {"kind": kind, "dtype": dtype, "tokens": _log(rng, 1 if kind == "linear" else 16,
                                                             600 if width == "14b" else 2048), "width": width}
        if kind == "linear":
            case["bias"] = rng.random() < 0.3
        return case
    if kind == "forward":
        return {"kind": kind, "dtype": "float32", "tokens": _log(rng, 16, 1500)}
    return {"kind": kind, "dtype": "float32", "tokens": _log(rng, 16, 1000), "new": rng.randint(8, 32)}


# ---------------------------------------------------------------------------------------------
# Inputs (plain torch, from the seed alone)
# ---------------------------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, std=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=g, device="cuda") * std).to(dtype)


def _dt(case):
    return torch.bfloat16 if case["dtype"] == "bfloat16" else torch.float32


def _inv_freq(d):
    return np.array([1.0 / (THETA ** (i / (d // 2))) for i in range(d // 2)], np.float64).astype(np.float32)


def _lens(case, seed):
    """Cached keys per sequence: a quarter of the longest and up, the longest among them."""
    r = np.random.RandomState(seed % (1 << 31))
    most = case["len"]
    lens = r.randint(max(1, most // 4), most + 1, size=case["batch"]).astype(np.int32)
    lens[r.randint(case["batch"])] = most
    return lens


def _inputs(case, seed):
    """The case's tensors as torch holds them (dict of torch tensors on the GPU)."""
    g, dt, bf = _gen(seed), _dt(case), torch.bfloat16
    kind = case["kind"]
    if kind == "attention":
        b, s, d = case["batch"], case["s"], case["d"]
        shape = (lambda h: (b, h, s, d)) if case["heads_first"] else (lambda h: (b, s, h, d))
        return {n: _randn(g, *shape(h), dtype=dt) for n, h in (("q", case["hq"]), ("k", case["hkv"]), ("v", case["hkv"]))}
    if kind == "decode":
        b, n, d = case["batch"], case["len"], case["d"]
        x = {"q": _randn(g, b, case["hq"], d, dtype=dt)}
        for name in ("k", "v"):
            x[name] = torch.stack([_randn(g, case["hkv"], n, d, dtype=dt) for _ in range(b)])
        return x
    h, i, hq, hkv = WIDTHS[case["width"]]
    d, m = 128, case["tokens"]
    if kind == "norm_rope":
        return {"x": _randn(g, m, h, dtype=dt), "w": 1 + _randn(g, h, std=0.1, dtype=dt), "q": _randn(g, 1, m, hq, d, dtype=dt),
                "k": _randn(g, 1, m, hkv, d, dtype=dt), "qw": 1 + _randn(g, d, std=0.1, dtype=dt),
                "kw": 1 + _randn(g, d, std=0.1, dtype=dt)}
    if kind == "qkv":
        return {"x": _randn(g, m, h, dtype=dt), "w": _randn(g, (hq + 2 * hkv) * d, h, std=0.02, dtype=bf),
                "qw": 1 + _randn(g, d, std=0.1, dtype=bf), "kw": 1 + _randn(g, d, std=0.1, dtype=bf)}
    if kind == "mlp":
        return {"x": _randn(g, m, h), "nw": 1 + _randn(g, h, std=0.1, dtype=dt), "gate": _randn(g, i, h, std=0.02, dtype=bf),
                "up": _randn(g, i, h, std=0.02, dtype=bf), "down": _randn(g, h, i, std=0.02, dtype=bf)}
    n = (hq + 2 * hkv) * d
    x = {"x": _randn(g, m, h, dtype=dt), "w": _randn(g, n, h, std=0.02, dtype=bf)}
    if case["bias"]:
        x["b"] = _randn(g, n, dtype=dt)
    return x


def _config():
    return Qwen3Config()


def _model_weights(seed):
    """(name, bf16 tensor on the GPU) of the model, one after another."""
    g, cfg = _gen(seed), _config()
    for name in weight_names(cfg):
        shape = weight_shape(cfg, name)
        norm = name.endswith("norm.weight")
        yield name, (1 + _randn(g, *shape, std=0.1)).to(torch.bfloat16) if norm else _randn(g, *shape, std=0.02, dtype=torch.bfloat16)


def _prompt(case, seed):
    return np.random.RandomState((seed + 77) % (1 << 31)).randint(0, VOCAB, size=case["tokens"]).astype(np.int32)


# ---------------------------------------------------------------------------------------------
# This framework's tensors seen by torch, and filled from it
# ---------------------------------------------------------------------------------------------
_NAME = {torch.float32: "float32", torch.bfloat16: "bfloat16", torch.int32: "int32"}
_CODE = {"float32": "<f4", "bfloat16": "<i2", "int32": "<i4"}


class _Device:
    """A contiguous tensor's device memory for torch.as_tensor (shared, not copied)."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.__cuda_array_interface__ = {"shape": tuple(tensor.shape), "typestr": _CODE[tensor.dtype], "strides": None,
                                         "data": (tensor.handle.data_ptr(), False), "version": 2}


def _seen(tensor):
    t = torch.as_tensor(_Device(tensor), device="cuda")
    return t.view(torch.bfloat16) if tensor.dtype == "bfloat16" else t


def _new(shape, dtype):
    return Tensor(shape=tuple(shape), dtype=dtype)


def _put(x):
    t = _new(x.shape, _NAME[x.dtype])
    _seen(t).copy_(x)
    return t


_ready = []


def _start():
    if not _ready:
        _ready.append(HipBackend.create(0))
    return env.get_backend("hip").operators


# ---------------------------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------------------------
def prepare(case, seed):
    ops = _start()
    kind = case["kind"]
    st = {"case": case}
    if kind in ("forward", "generate"):
        weights = {n: w.view(torch.int16).cpu().numpy().view(np.uint16) for n, w in _model_weights(seed)}
        room = -(-(case["tokens"] + case.get("new", 0)) // 256) * 256
        st["model"] = Qwen3ForCausalLM(_config(), weights, max_seq_len=room, activations=case["dtype"])
        st["prompt"] = _prompt(case, seed)
        return st
    x = _inputs(case, seed)
    t = st["t"] = {n: _put(v) for n, v in x.items() if n not in ("gate", "up")}
    outs = {}
    if kind == "attention":
        if not case["heads_first"]:
            for n in ("q", "k", "v"):
                t[n] = F.permute(t[n], (0, 2, 1, 3))
        outs["o"] = _new((case["batch"], case["hq"], case["s"], case["d"]), case["dtype"])
        st["kernel"] = ops.find("flash_attention_split")
    elif kind == "decode":
        t["lens"] = Tensor(_lens(case, seed), dtype="int32")
        outs["o"] = _new(t["q"].shape, case["dtype"])
        st["kernel"] = ops.find("decode_attention")
    elif kind == "norm_rope":
        m = case["tokens"]
        h, _, hq, hkv = WIDTHS[case["width"]]
        t["inv"] = Tensor(_inv_freq(128), dtype="float32")
        t["pos"] = Tensor(np.arange(m, dtype=np.int32), dtype="int32")
        outs = {"y": _new((m, h), case["dtype"]), "q": _new((1, hq, m, 128), case["dtype"]),
                "k": _new((1, hkv, m, 128), case["dtype"])}
        st["norm"], st["rope"] = ops.find("rms_norm"), ops.find("rms_norm_rope")
    elif kind == "qkv":
        m = case["tokens"]
        _, _, hq, hkv = WIDTHS[case["width"]]
        t["inv"] = Tensor(_inv_freq(128), dtype="float32")
        t["pos"] = Tensor(np.arange(m, dtype=np.int32), dtype="int32")
        outs = {n: _new((1, k, m, 128), case["dtype"]) for n, k in (("q", hq), ("k", hkv), ("v", hkv))}
        st["kernel"], st["table"] = ops.find("linear_qk_norm_rope"), ops.find("rope_table")
        st["table_out"] = _new((m, 64, 2), "float32")
    elif kind == "mlp":
        # gate and up rows interleaved in blocks of 8, the layout linear_swiglu documents
        i, h = x["gate"].shape
        t["gu"] = _put(torch.stack([x["gate"].view(i // 8, 8, h), x["up"].view(i // 8, 8, h)], 1).reshape(2 * i, h))
        outs["y"] = _new((case["tokens"], h), "float32")
    else:
        outs["y"] = _new((case["tokens"], x["w"].shape[0]), case["dtype"])
    st["outs"], st["seen"] = outs, {n: _seen(o) for n, o in outs.items()}
    torch.cuda.synchronize()
    return st


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "forward":
        return _seen(state["model"].forward(state["prompt"], 0))
    if kind == "generate":
        tokens, logits = state["model"].generate(state["prompt"], case["new"], return_logits=True)
        return {"tokens": np.asarray(tokens, np.int64), "logits": logits}
    t, outs = state["t"], state["outs"]
    if kind == "attention":
        if case["split"]:
            state["kernel"](t["q"].handle, t["k"].handle, t["v"].handle, outs["o"].handle, 1.0 / math.sqrt(case["d"]),
                            case["causal"])
        else:
            F.scaled_dot_product_attention(t["q"], t["k"], t["v"], is_causal=case["causal"], out=outs["o"])
    elif kind == "decode":
        state["kernel"](t["q"].handle, t["k"].handle, t["v"].handle, t["lens"].handle, outs["o"].handle,
                        1.0 / math.sqrt(case["d"]))
    elif kind == "norm_rope":
        state["norm"]([t["x"].handle], {"normalized_shape": [t["x"].shape[-1]], "eps": EPS, "weight": t["w"].handle,
                                        "out": outs["y"].handle})
        state["rope"](t["q"].handle, t["k"].handle, {"q_weight": t["qw"].handle, "k_weight": t["kw"].handle,
                                                     "inv_freq": t["inv"].handle, "positions": t["pos"].handle,
                                                     "eps": EPS, "q_out": outs["q"].handle, "k_out": outs["k"].handle})
    elif kind == "qkv":
        table = state["table"](t["pos"].handle, t["inv"].handle, state["table_out"].handle)
        state["kernel"](t["x"].handle, t["w"].handle, {"q_weight": t["qw"].handle, "k_weight": t["kw"].handle,
                                                       "inv_freq": t["inv"].handle, "positions": t["pos"].handle,
                                                       "eps": EPS, "q_out": outs["q"].handle, "k_out": outs["k"].handle,
                                                       "v_out": outs["v"].handle, "rope_table": table})
    elif kind == "mlp":
        h = F.rms_norm(t["x"], [t["x"].shape[-1]], t["nw"], EPS, out_dtype=case["dtype"])
        a = F.linear_swiglu(h, t["gu"])
        F.dispatch_matmul(a, t["down"], c=t["x"], beta=1.0, out=outs["y"], transpose_b=True)
    else:
        F.dispatch_matmul(t["x"], t["w"], bias=t.get("b"), out=outs["y"], transpose_b=True)
    return state["seen"]


# ---------------------------------------------------------------------------------------------
# work / tolerance / exact
# ---------------------------------------------------------------------------------------------
def _model_work(tokens, new):
    h, i, hq, hkv = WIDTHS["0.6b"]
    layer = h * (hq + 2 * hkv) * 128 + hq * 128 * h + 3 * h * i
    prefill = 28 * (2 * layer * tokens + 4 * 128 * hq * tokens * tokens / 2) + 2 * VOCAB * h
    weights = 2 * (28 * layer + VOCAB * h)
    row = 28 * 2 * hkv * 128 * 4  # K and V of one token, float32
    step = 2 * (28 * layer + VOCAB * h)
    attended = sum(tokens + j + 1 for j in range(new))
    return {"bytes": weights * (1 + new) + row * (tokens + attended + new) + 4 * VOCAB * (1 + new),
            "flops": prefill + new * step + 28 * 4 * 128 * hq * attended}


def work(case):
    kind = case["kind"]
    size = 2 if case["dtype"] == "bfloat16" else 4
    if kind in ("forward", "generate"):
        return _model_work(case["tokens"], case.get("new", 0))
    if kind == "attention":
        b, s, d, hq, hkv = case["batch"], case["s"], case["d"], case["hq"], case["hkv"]
        pairs = s * (s + 1) / 2 if case["causal"] else s * s
        return {"bytes": size * b * s * d * (2 * hq + 2 * hkv), "flops": 4 * d * b * hq * pairs}
    if kind == "decode":
        # the mean of _lens
        keys = case["len"] + (case["batch"] - 1) * (case["len"] + max(1, case["len"] // 4)) / 2
        return {"bytes": size * (2 * keys * case["hkv"] * case["d"] + 2 * case["batch"] * case["hq"] * case["d"]),
                "flops": 4 * keys * case["hq"] * case["d"]}
    h, i, hq, hkv = WIDTHS[case["width"]]
    m, n = case["tokens"], (hq + 2 * hkv) * 128
    if kind == "norm_rope":
        return {"bytes": size * 2 * m * (h + (hq + hkv) * 128), "flops": m * (4 * h + 10 * (hq + hkv) * 128)}
    if kind == "mlp":
        return {"bytes": 2 * 3 * h * i + 4 * 2 * m * h, "flops": 2 * m * 3 * h * i}
    return {"bytes": 2 * n * h + size * m * (h + n), "flops": 2 * m * n * h}


def tolerance(case):
    """Relative errors (2-norm) that another order of the sums, or another tiling of them, may show."""
    if case["dtype"] == "bfloat16":
        # outputs (and the weights of attention, the intermediates of the MLP) are rounded to 2^-9
        return {"rel": 1e-2, "max": 0.1}
    if case["kind"] in ("forward", "generate"):
        # differences of 2^-17 in each product travel through 28 layers: 8e-6 against float64
        return {"rel": 4e-5, "max": 2e-3}
    # float32 activations are multiplied as a bf16 pair (2^-17 each), float32 sums: 2e-6 to 5e-6 against float64
    return {"rel": 2e-5, "max": 1e-3}


def _rms(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w


def _rope(x, m, start=0):
    """x [..., m, d]; the angle is the float32 product of position and frequency, as RoPE defines it here."""
    pos = torch.arange(start, start + m, device=x.device, dtype=torch.float32)
    ang = (pos[:, None] * torch.from_numpy(_inv_freq(x.shape[-1])).to(x.device)[None]).double()
    c, s = torch.cat([ang.cos()] * 2, -1), torch.cat([ang.sin()] * 2, -1)
    a, b = x.chunk(2, -1)
    return x * c + torch.cat([-b, a], -1) * s


def _attend(q, k, v, causal):
    """[h, l, d], [g, s, d] in float64; query i is the key length's i-th from the end when causal."""
    out = []
    ratio = q.shape[0] // k.shape[0]
    for h in range(q.shape[0]):
        sc = q[h] @ k[h // ratio].t() / math.sqrt(q.shape[-1])
        if causal:
            lq, lk = sc.shape
            sc.masked_fill_(torch.ones(lq, lk, dtype=torch.bool, device=sc.device).triu(lk - lq + 1), -math.inf)
        out.append(torch.softmax(sc, -1) @ v[h // ratio])
    return torch.stack(out)


def _model_exact(case, seed):
    cfg = _config()
    w = dict(_model_weights(seed))
    hq, hkv, d = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim
    cache = [None] * cfg.num_hidden_layers

    def forward(ids, start):
        x = w["model.embed_tokens.weight"][torch.from_numpy(np.asarray(ids, np.int64)).cuda()].double()
        m = x.shape[0]
        for li in range(cfg.num_hidden_layers):
            p = "model.layers.%d." % li
            g = lambda n: w[p + n + ".weight"].double()  # noqa: E731
            h = _rms(x, g("input_layernorm"))
            heads = lambda n, c: (h @ g("self_attn." + n).t()).view(m, c, d).transpose(0, 1)  # noqa: E731
            q = _rope(_rms(heads("q_proj", hq), g("self_attn.q_norm")), m, start)
            k = _rope(_rms(heads("k_proj", hkv), g("self_attn.k_norm")), m, start)
            v = heads("v_proj", hkv)
            if cache[li] is not None:
                k, v = torch.cat([cache[li][0], k], 1), torch.cat([cache[li][1], v], 1)
            cache[li] = (k, v)
            x = x + _attend(q, k, v, m > 1).transpose(0, 1).reshape(m, hq * d) @ g("self_attn.o_proj").t()
            h = _rms(x, g("post_attention_layernorm"))
            x = x + (torch.nn.functional.silu(h @ g("mlp.gate_proj").t()) * (h @ g("mlp.up_proj").t())) @ g("mlp.down_proj").t()
        return _rms(x[-1:], w["model.norm.weight"].double()) @ w["model.embed_tokens.weight"].double().t()

    logits = [forward(_prompt(case, seed), 0)]
    if case["kind"] == "forward":
        return logits[0]
    tokens = []
    for j in range(case["new"]):
        tokens.append(int(logits[-1].argmax()))
        logits.append(forward([tokens[-1]], case["tokens"] + j))
    return {"tokens": None, "logits": [x[0] for x in logits]}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("forward", "generate"):
        return _model_exact(case, seed)
    x = _inputs(case, seed)
    if kind == "attention":
        if not case["heads_first"]:
            x = {n: v.transpose(1, 2) for n, v in x.items()}
        return {"o": torch.stack([_attend(*(x[n][b].double() for n in ("q", "k", "v")), case["causal"])
                                  for b in range(case["batch"])])}
    if kind == "decode":
        out = []
        for b, n in enumerate(_lens(case, seed).tolist()):
            out.append(_attend(x["q"][b].double()[:, None], x["k"][b, :, :n].double(), x["v"][b, :, :n].double(), False)[:, 0])
        return {"o": torch.stack(out)}
    x = {n: v.double() for n, v in x.items()}
    m = case["tokens"]
    if kind == "norm_rope":
        return {"y": _rms(x["x"], x["w"]), "q": _rope(_rms(x["q"], x["qw"]).transpose(1, 2), m),
                "k": _rope(_rms(x["k"], x["kw"]).transpose(1, 2), m)}
    if kind == "qkv":
        _, _, hq, hkv = WIDTHS[case["width"]]
        y = (x["x"] @ x["w"].t()).view(1, m, hq + 2 * hkv, 128).transpose(1, 2)
        return {"q": _rope(_rms(y[:, :hq], x["qw"]), m), "k": _rope(_rms(y[:, hq:hq + hkv], x["kw"]), m), "v": y[:, hq + hkv:]}
    if kind == "mlp":
        h = _rms(x["x"], x["nw"])
        return {"y": x["x"] + (torch.nn.functional.silu(h @ x["gate"].t()) * (h @ x["up"].t())) @ x["down"].t()}
    y = x["x"] @ x["w"].t()
    return {"y": y + x["b"] if "b" in x else y}
