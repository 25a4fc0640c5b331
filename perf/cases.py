"""What a program that uses this framework has it do, as cases that can be timed and checked.

Whole calls (a short generation, one decode step, one prompt prefill) go
through ``LlamaModel``; single layers and blocks go through the C ABI that a
host program links against (``ammon_amd._abi``), on buffers that are torch
tensors.  Sizes are those of this repository's benchmark and tests: the
stories15M-shaped fp32 decoder, the Llama-3-8B shape, one Llama-3-70B-shaped
layer, and ragged sizes between them.
"""
import ctypes
import math

import numpy as np
import torch

import ammon_amd
from ammon_amd import _abi
from ammon_amd._abi import BF16, F32, call

STORIES = dict(dim=288, layers=6, heads=6, kv_heads=6, hidden=768, vocab=32000, theta=10000.0,
               w="f32", kv="f32")
LLAMA8B = dict(dim=4096, layers=32, heads=32, kv_heads=8, hidden=14336, vocab=128256,
               theta=500000.0, w="bf16", kv="bf16")
EPS = 1e-5


def listed():
    return [
        # a short story from the small fp32 model, greedily on the device: every launch is tiny
        dict(STORIES, name="generate_stories", kind="generate", seq=256, prompt=8, new=64),
        # the same model's prompt before the first token: small fp32 GEMMs
        dict(STORIES, name="prefill_stories", kind="prefill", seq=256, start=0, tokens=100),
        # one token of the 8B shape at the end of an 8k context, logits to the host: the headline
        dict(LLAMA8B, name="step_8b_ctx8k", kind="step", seq=8192, pos=8150),
        # a document-sized prompt of the 8B shape, whole model
        dict(LLAMA8B, name="prefill_8b_1000", kind="prefill", seq=8192, start=0, tokens=1000),
        # decode attention of one layer: 8B heads over the reference's fp32 cache, mid context
        dict(name="attn_fp32_ctx4k", kind="attn", heads=32, kv_heads=8, head=128, seq=8192, pos=4000,
             kv="f32"),
        # ... and the 70B-shaped layer over a full 32k bf16 cache
        dict(name="attn_70b_ctx32k", kind="attn", heads=64, kv_heads=8, head=128, seq=32768,
             pos=32760, kv="bf16"),
        # the 70B-shaped layer's SwiGLU block for one token
        dict(name="mlp_70b_decode", kind="mlp", dim=8192, hidden=28672, tokens=1, w="bf16"),
        # prompt attention of one 8B layer: a whole 2k prompt ...
        dict(name="prefill_attn_2k", kind="prefill_attn", heads=32, kv_heads=8, head=128, seq=8192,
             start=0, tokens=2048, kv="bf16"),
        # ... and a follow-up turn of odd length late in a long chat
        dict(name="prefill_attn_turn", kind="prefill_attn", heads=32, kv_heads=8, head=128, seq=8192,
             start=7001, tokens=301, kv="bf16"),
        # the 8B SwiGLU block for a one-line prompt: weights streamed for 16 tokens
        dict(name="mlp_8b_16", kind="mlp", dim=4096, hidden=14336, tokens=16, w="bf16"),
        # ... and for a long prompt: compute on the matrix cores
        dict(name="mlp_8b_2k", kind="mlp", dim=4096, hidden=14336, tokens=2048, w="bf16"),
        # the 8B attention block's front for a paragraph of odd length
        dict(name="qkv_8b_131", kind="qkv", dim=4096, heads=32, kv_heads=8, head=128, seq=8192,
             start=77, tokens=131, w="bf16", kv="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["generate", "prefill", "step", "attn", "attn", "prefill_attn",
                       "prefill_attn", "mlp", "mlp", "qkv"])
    heads, kv_heads, head = rng.choice([(32, 8, 128), (64, 8, 128), (32, 8, 128), (16, 16, 128),
                                        (24, 12, 128), (32, 8, 64), (18, 6, 96), (8, 8, 48),
                                        (4, 1, 80)])
    w, kv = rng.choice(["bf16", "bf16", "f32"]), rng.choice(["bf16", "bf16", "f32"])
    if kind in ("generate", "prefill", "step"):
        heads, kv_heads, head = rng.choice([(6, 6, 48), (8, 4, 64), (8, 2, 128), (16, 4, 128)])
        c = dict(kind=kind, dim=heads * head, layers=rng.randint(2, 6), heads=heads,
                 kv_heads=kv_heads, hidden=8 * _log(rng, 64, 700), vocab=_log(rng, 2000, 64000),
                 theta=rng.choice([10000.0, 500000.0]), w=w, kv=kv)
        if kind == "generate":
            c.update(seq=512, kv="f32", prompt=_log(rng, 1, 64), new=_log(rng, 66, 160))
        elif kind == "prefill":
            start = rng.choice([0, 0, _log(rng, 1, 2000)])
            c.update(seq=4096, start=start, tokens=_log(rng, 2, 1500))
        else:
            c.update(seq=4096, pos=_log(rng, 4, 4095))
        return c
    if kind == "attn":
        seq = rng.choice([1024, 8192, 32768])
        return dict(kind=kind, heads=heads, kv_heads=kv_heads, head=head, seq=seq,
                    pos=_log(rng, 16, seq - 1), kv=kv)
    if kind == "prefill_attn":
        return dict(kind=kind, heads=heads, kv_heads=kv_heads, head=head, seq=8192,
                    start=rng.choice([0, 0, _log(rng, 1, 6000)]), tokens=_log(rng, 2, 2000), kv=kv)
    if kind == "mlp":
        dim = 8 * _log(rng, 36, 1024)
        return dict(kind=kind, dim=dim, hidden=8 * _log(rng, 90, 3584),
                    tokens=rng.choice([1, _log(rng, 2, 2000), _log(rng, 2, 2000)]), w=w)
    dim = 8 * _log(rng, 36, 1024)
    return dict(kind=kind, dim=dim, heads=heads, kv_heads=kv_heads, head=head, seq=4096,
                start=rng.choice([0, _log(rng, 1, 2000)]), tokens=_log(rng, 2, 2000), w=w, kv=kv)


# ---- inputs -----------------------------------------------------------------------------------
_RUNTIME = None


def _rt():
    global _RUNTIME
    if _RUNTIME is None:
        _RUNTIME = ammon_amd.Runtime(0)
    return _RUNTIME


def _dt(name):
    return torch.bfloat16 if name == "bf16" else torch.float32


def _ab(name):
    return BF16 if name == "bf16" else F32


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


class _Draws:
    """Seeded normal tensors on the GPU, in the order they are asked for."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, shape, std=1.0, dtype=torch.float32, mean=0.0):
        return torch.empty(shape, dtype=dtype, device="cuda").normal_(mean, std, generator=self.g)

    def ids(self, n, vocab):
        return torch.randint(0, vocab, (n,), generator=self.g, device="cuda").cpu().numpy().astype(
            np.int32)


def _model_inputs(c, seed):
    """Stacked weights, the cache (positions before the call; NULL for a fresh one) and token ids."""
    d, wd = _Draws(seed), _dt(c["w"])
    L, dim, hid = c["layers"], c["dim"], c["hidden"]
    head = dim // c["heads"]
    q, k = head * c["heads"], head * c["kv_heads"]
    std = 0.02 if dim >= 1024 else 0.05
    w = {
        "tok_emb": d.normal((c["vocab"], dim), std, wd),
        "rms_att": d.normal((L, dim), 0.1, mean=1.0), "rms_ffn": d.normal((L, dim), 0.1, mean=1.0),
        "wq": d.normal((L, q, dim), std, wd), "wk": d.normal((L, k, dim), std, wd),
        "wv": d.normal((L, k, dim), std, wd), "wo": d.normal((L, dim, q), std, wd),
        "w1": d.normal((L, hid, dim), std, wd), "w2": d.normal((L, dim, hid), std, wd),
        "w3": d.normal((L, hid, dim), std, wd), "rms_final": d.normal((dim,), 0.1, mean=1.0),
        "wcls": d.normal((c["vocab"], dim), std, wd),
    }
    past = {"generate": 0, "prefill": c.get("start", 0), "step": c.get("pos", 0)}[c["kind"]]
    cache = None
    if past:
        cache = d.normal((2, L, c["kv_heads"], c["seq"], head), 1.0, _dt(c["kv"]))
    n = {"generate": c.get("prompt"), "prefill": c.get("tokens"), "step": 1}[c["kind"]]
    return w, cache, past, d.ids(n, c["vocab"])


class _Config:
    def __init__(self, c):
        self.dim, self.n_layers, self.n_heads = c["dim"], c["layers"], c["heads"]
        self.n_kv_heads, self.hidden, self.vocab = c["kv_heads"], c["hidden"], c["vocab"]
        self.max_seq, self.theta, self.eps = c["seq"], c["theta"], EPS
        self.w_dtype, self.kv_dtype = _ab(c["w"]), _ab(c["kv"])


class _View:
    """The model's own device memory, for torch.as_tensor."""

    def __init__(self, ptr, shape, bf16):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "version": 2,
                                         "typestr": "<i2" if bf16 else "<f4", "strides": None}


def _kv_views(m, c, layer):
    k, v = ctypes.c_void_p(), ctypes.c_void_p()
    call("ammon_llama_kv_layer", m.handle, layer, ctypes.byref(k), ctypes.byref(v))
    shape, bf = (c["kv_heads"], c["seq"], c["dim"] // c["heads"]), c["kv"] == "bf16"
    out = [torch.as_tensor(_View(p.value, shape, bf), device="cuda") for p in (k, v)]
    out = [t.view(torch.bfloat16) if bf else t for t in out]
    for t in out:
        t.model = m  # the memory is the model's: it lives as long as the tensor does
    return out


def _rope_table(theta, head, seq):
    """[seq, head / 2, 2]: the fp32 angles of the reference (1 / powf(theta, hd / head), times the
    position), then cos and sin."""
    powf = ctypes.CDLL("libm.so.6").powf
    powf.restype, powf.argtypes = ctypes.c_float, [ctypes.c_float, ctypes.c_float]
    freq = np.array([np.float32(1.0) / np.float32(powf(theta, np.float32(h) / np.float32(head)))
                     for h in range(0, head, 2)], np.float32)
    ang = (np.arange(seq, dtype=np.float32)[:, None] * freq[None, :]).astype(np.float64)
    return np.stack([np.cos(ang), np.sin(ang)], -1)


def _layer_inputs(c, seed):
    d = _Draws(seed)
    if c["kind"] in ("attn", "prefill_attn"):
        n = c.get("tokens", 1)
        kv = d.normal((2, c["kv_heads"], c["seq"], c["head"]), 1.0, _dt(c["kv"]))
        return {"q": d.normal((n, c["heads"], c["head"])), "k": kv[0], "v": kv[1]}
    wd, std, dim = _dt(c["w"]), 0.02, c["dim"]
    t = {"x": d.normal((c["tokens"], dim)), "norm": d.normal((dim,), 0.1, mean=1.0)}
    if c["kind"] == "mlp":
        t.update(w1=d.normal((c["hidden"], dim), std, wd), w3=d.normal((c["hidden"], dim), std, wd),
                 w2=d.normal((dim, c["hidden"]), std, wd))
    else:
        q, k = c["heads"] * c["head"], c["kv_heads"] * c["head"]
        t.update(wq=d.normal((q, dim), std, wd), wk=d.normal((k, dim), std, wd),
                 wv=d.normal((k, dim), std, wd))
    return t


def _split_len(c):
    """The split a program takes: the library's own for decode; for a prompt, as many units as the
    device holds twice (the model's rule)."""
    rt, lib = _rt(), _abi.lib
    if c["kind"] == "attn":
        return int(lib.ammon_attention_default_split_for(rt.handle, c["heads"], c["kv_heads"],
                                                         c["head"], _ab(c["kv"]), c["seq"]))
    split, ctx = 16, c["start"] + c["tokens"]
    while split < 1024 and c["kv_heads"] * c["tokens"] * int(
            lib.ammon_attention_splits(ctx, split)) > 2 * rt.info.compute_units:
        split *= 2
    return split


def prepare(case, seed):
    c, rt = case, _rt()
    if c["kind"] in ("generate", "prefill", "step"):
        w, cache, past, ids = _model_inputs(c, seed)
        m = ammon_amd.LlamaModel(rt, _Config(c), {n: t.data_ptr() for n, t in w.items()})
        for layer in range(c["layers"]):
            for side, view in enumerate(_kv_views(m, c, layer)):
                if cache is None:
                    view.zero_()
                else:
                    view.copy_(cache[side, layer])
        torch.cuda.synchronize()
        return {"c": c, "w": w, "m": m, "ids": ids, "kv": _kv_views(m, c, c["layers"] - 1)}
    t = _layer_inputs(c, seed)
    s = {"c": c, "t": t}
    empty = lambda *shape: torch.empty(shape, device="cuda")  # noqa: E731
    if c["kind"] in ("attn", "prefill_attn"):
        s["split"] = _split_len(c)
        n = c.get("tokens", 1)
        if c["kind"] == "attn":
            nbytes = int(_abi.lib.ammon_attention_scratch_bytes(c["heads"], c["head"], c["seq"],
                                                                s["split"]))
        else:
            nbytes = int(_abi.lib.ammon_attention_prefill_scratch_bytes(
                n, c["heads"], c["head"], c["start"] + n, s["split"]))
        s["part"], s["part_bytes"] = empty(nbytes // 4), nbytes
        s["out"] = torch.empty_like(t["q"])
        s["step"] = torch.tensor([0, c.get("pos", c.get("start"))], dtype=torch.int32, device="cuda")
        return s
    n, dim = c["tokens"], c["dim"]
    s["xn"] = empty(n, dim)
    if c["kind"] == "mlp":
        s["hb"], s["y"], rows = empty(n, c["hidden"]), empty(n, dim), dim
    else:
        q, k = c["heads"] * c["head"], c["kv_heads"] * c["head"]
        rows = q + 2 * k
        s["q"] = empty(n, q)
        s["k"], s["v"] = (torch.zeros((c["kv_heads"], c["seq"], c["head"]), dtype=_dt(c["kv"]),
                                      device="cuda") for _ in range(2))
        s["table"] = torch.from_numpy(_rope_table(10000.0, c["head"], c["seq"]).astype(
            np.float32)).cuda()
        s["step"] = torch.tensor([0, c["start"]], dtype=torch.int32, device="cuda")
    s["ws_bytes"] = int(_abi.lib.ammon_prefill_gemm_workspace_bytes(rows, n))
    s["ws"] = empty(s["ws_bytes"] // 4)
    return s


# ---- one pass -----------------------------------------------------------------------------------
def run(state):
    s, c = state, state["c"]
    if c["kind"] == "generate":
        tokens, logits, _ = s["m"].generate_tokens_device(s["ids"], c["new"])
        return {"tokens": tokens, "logits": logits, "k": s["kv"][0], "v": s["kv"][1]}
    if c["kind"] == "prefill":
        logits = s["m"].prefill(s["ids"], c["start"])
        return {"logits": logits, "k": s["kv"][0], "v": s["kv"][1]}
    if c["kind"] == "step":
        logits = s["m"].step(int(s["ids"][0]), c["pos"])
        return {"logits": logits, "k": s["kv"][0], "v": s["kv"][1]}
    h, t = _rt().handle, s["t"]
    if c["kind"] == "attn":
        call("ammon_attention_decode", h, None, _p(t["q"]), c["heads"], _p(t["k"]), _p(t["v"]),
             _ab(c["kv"]), c["kv_heads"], c["head"], c["seq"], _p(s["step"]), s["split"],
             _p(s["part"]), s["part_bytes"], _p(s["out"]))
        return s["out"]
    if c["kind"] == "prefill_attn":
        call("ammon_attention_prefill", h, None, _p(t["q"]), c["tokens"], c["heads"], _p(t["k"]),
             _p(t["v"]), _ab(c["kv"]), c["kv_heads"], c["head"], c["seq"], _p(s["step"]),
             c["start"] + c["tokens"], s["split"], _p(s["part"]), s["part_bytes"], _p(s["out"]))
        return s["out"]
    n, dim = c["tokens"], c["dim"]
    if c["kind"] == "mlp" and n == 1:
        call("ammon_gate_up_swiglu", h, None, _p(t["x"]), _p(t["norm"]), F32, EPS, _p(t["w1"]),
             _p(t["w3"]), _ab(c["w"]), dim, c["hidden"], _p(s["hb"]))
        call("ammon_gemv", h, None, _p(t["w2"]), _ab(c["w"]), dim, c["hidden"], _p(s["hb"]),
             _p(s["y"]), _p(t["x"]))
        return [s["hb"], s["y"]]
    call("ammon_rmsnorm", h, None, _p(t["x"]), _p(t["norm"]), F32, _p(s["xn"]), n, dim, EPS)
    if c["kind"] == "mlp":
        call("ammon_prefill_gate_up_swiglu", h, None, _p(s["xn"]), n, _p(t["w1"]), _p(t["w3"]),
             _ab(c["w"]), dim, c["hidden"], _p(s["hb"]))
        call("ammon_prefill_gemm_ws", h, None, _p(t["w2"]), _ab(c["w"]), dim, c["hidden"],
             _p(s["hb"]), n, _p(s["y"]), _p(t["x"]), _p(s["ws"]), s["ws_bytes"])
        return [s["hb"], s["y"]]
    call("ammon_prefill_qkv_rope_store_ws", h, None, _p(s["xn"]), n, _p(t["wq"]), _p(t["wk"]),
         _p(t["wv"]), _ab(c["w"]), dim, c["heads"], c["kv_heads"], c["head"], _p(s["q"]),
         _p(s["k"]), _p(s["v"]), _ab(c["kv"]), c["seq"], _p(s["step"]), _p(s["table"]), _p(s["ws"]),
         s["ws_bytes"])
    return [s["q"], s["k"], s["v"]]


# ---- what a pass cannot do without ---------------------------------------------------------------
def _size(name):
    return 2 if name == "bf16" else 4


def work(case):
    c = case
    n = c.get("tokens", 1)
    if c["kind"] in ("generate", "prefill", "step"):
        head = c["dim"] // c["heads"]
        q, kv = head * c["heads"], head * c["kv_heads"]
        layer = (q + 2 * kv) * c["dim"] + c["dim"] * q + 3 * c["hidden"] * c["dim"]
        weights = (c["layers"] * layer + c["vocab"] * c["dim"]) * _size(c["w"])
        passes, first = {"generate": (c.get("new", 1) - 1, 0), "prefill": (1, c.get("start", 0)),
                         "step": (1, c.get("pos", 0))}[c["kind"]]
        rows = passes if c["kind"] == "generate" else n
        pairs = sum(first + i + 1 for i in range(rows))  # (query, key) pairs of one head
        read = pairs if c["kind"] == "generate" else first + n
        kv_bytes = c["layers"] * 2 * kv * _size(c["kv"]) * (read + rows)
        flops = 2 * rows * c["layers"] * layer + 4 * c["layers"] * q * pairs + \
            2 * passes * c["vocab"] * c["dim"]
        return {"bytes": passes * weights + kv_bytes + passes * 4 * c["vocab"], "flops": flops}
    if c["kind"] in ("attn", "prefill_attn"):
        first = c.get("pos", c.get("start"))
        pairs = sum(first + i + 1 for i in range(n))
        kv = 2 * c["kv_heads"] * c["head"] * (first + n) * _size(c["kv"])
        return {"bytes": kv + 8 * n * c["heads"] * c["head"],
                "flops": 4 * c["heads"] * c["head"] * pairs}
    if c["kind"] == "mlp":
        w = 3 * c["dim"] * c["hidden"]
        return {"bytes": w * _size(c["w"]) + 4 * n * (2 * c["dim"] + c["hidden"]), "flops": 2 * n * w}
    q, kv = c["heads"] * c["head"], c["kv_heads"] * c["head"]
    w = (q + 2 * kv) * c["dim"]
    return {"bytes": w * _size(c["w"]) + 4 * n * (c["dim"] + q) + 2 * n * kv * _size(c["kv"]),
            "flops": 2 * n * w}


# About four times what this implementation is off from exact() or from itself with its sums in
# another order.  A bf16 cache rounds each stored key and value, and fp32 sums in another order move
# some of them by one step of bf16 (2^-8): stored rows then differ by that in a few places, and what
# is computed from them by a little in every place.
def tolerance(case):
    stored = case.get("kv") == "bf16"
    if case["kind"] in ("generate", "prefill", "step"):
        return {"rel": 1e-2, "max": 0.1} if stored else {"rel": 1e-4, "max": 4e-3}
    if case["kind"] == "qkv" and stored:
        return {"rel": 1e-3, "max": 0.05}
    return {"rel": 1e-5, "max": 4e-4}


# ---- the same in 64 bits ---------------------------------------------------------------------------
def _d(t):
    return t.to(torch.float64)


def _norm(x, w):
    return _d(w) * x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)


def _rotate(x, table, first):
    """x [n, heads, head] at positions first..: pairs (2i, 2i + 1)."""
    cs = table[first:first + x.shape[0]][:, None]
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * cs[..., 0] - b * cs[..., 1], a * cs[..., 1] + b * cs[..., 0]],
                       -1).reshape(x.shape)


def _attend(q, k, v, first):
    """q [n, heads, head] at positions first.. over k, v [kv_heads, seq, head]."""
    n, heads, head = q.shape
    out = torch.empty_like(q)
    g, ctx = heads // k.shape[0], first + n
    at = torch.arange(first, ctx, device="cuda")[:, None]
    late = torch.arange(ctx, device="cuda")[None, :] > at
    for h in range(heads):
        kk, vv = _d(k[h // g, :ctx]), _d(v[h // g, :ctx])
        s = (q[:, h] @ kk.t()) / math.sqrt(head)
        out[:, h] = torch.softmax(s.masked_fill(late, -math.inf), -1) @ vv
    return out


def _forward(c, w, cache, ids, first, table):
    """Logits of the last of `ids` at positions first.. in float64; the cache [2, L, kv_heads, seq,
    head] takes their rows in its own type."""
    head = c["dim"] // c["heads"]
    x = _d(w["tok_emb"][torch.from_numpy(np.asarray(ids, np.int64)).cuda()])
    n = x.shape[0]
    for l in range(c["layers"]):
        xn = _norm(x, w["rms_att"][l])
        q = _rotate((xn @ _d(w["wq"][l]).t()).reshape(n, -1, head), table, first)
        k = _rotate((xn @ _d(w["wk"][l]).t()).reshape(n, -1, head), table, first)
        v = (xn @ _d(w["wv"][l]).t()).reshape(n, -1, head)
        cache[0, l][:, first:first + n] = k.transpose(0, 1).to(cache.dtype)
        cache[1, l][:, first:first + n] = v.transpose(0, 1).to(cache.dtype)
        a = _attend(q, cache[0, l], cache[1, l], first).reshape(n, -1)
        x = x + a @ _d(w["wo"][l]).t()
        xn = _norm(x, w["rms_ffn"][l])
        g = xn @ _d(w["w1"][l]).t()
        x = x + (g * torch.sigmoid(g) * (xn @ _d(w["w3"][l]).t())) @ _d(w["w2"][l]).t()
    return _norm(x[-1], w["rms_final"]) @ _d(w["wcls"]).t()


def exact(case, seed):
    c = case
    if c["kind"] in ("generate", "prefill", "step"):
        w, cache, past, ids = _model_inputs(c, seed)
        head = c["dim"] // c["heads"]
        if cache is None:
            cache = torch.zeros((2, c["layers"], c["kv_heads"], c["seq"], head), device="cuda",
                                dtype=torch.float64 if c["kv"] == "f32" else torch.bfloat16)
        elif c["kv"] == "f32":
            cache = _d(cache)
        table = torch.from_numpy(_rope_table(c["theta"], head, c["seq"])).cuda()
        if c["kind"] != "generate":
            logits = _forward(c, w, cache, ids, past, table)
        else:
            tok = int(ids[0])
            for pos in range(c["new"] - 1):
                logits = _forward(c, w, cache, [tok], pos, table)
                tok = int(ids[pos + 1]) if pos + 1 < len(ids) else int(logits.argmax())
        k, v = cache[0, -1], cache[1, -1]
        out = {"logits": logits, "k": k, "v": v}
        return dict(out, tokens=None) if c["kind"] == "generate" else out
    t = _layer_inputs(c, seed)
    if c["kind"] in ("attn", "prefill_attn"):
        return _attend(_d(t["q"]), t["k"], t["v"], c.get("pos", c.get("start")))
    x = _d(t["x"])
    xn = _norm(x, t["norm"])
    if c["kind"] == "mlp":
        g = xn @ _d(t["w1"]).t()
        hb = g * torch.sigmoid(g) * (xn @ _d(t["w3"]).t())
        return [hb, x + hb @ _d(t["w2"]).t()]
    n, first = c["tokens"], c["start"]
    table = torch.from_numpy(_rope_table(10000.0, c["head"], c["seq"])).cuda()
    rows = lambda m: (xn @ _d(m).t()).reshape(n, -1, c["head"])  # noqa: E731
    k, v = (torch.zeros((c["kv_heads"], c["seq"], c["head"]), device="cuda",
                        dtype=torch.float64 if c["kv"] == "f32" else torch.bfloat16)
            for _ in range(2))
    k[:, first:first + n] = _rotate(rows(t["wk"]), table, first).transpose(0, 1).to(k.dtype)
    v[:, first:first + n] = rows(t["wv"]).transpose(0, 1).to(v.dtype)
    return [_rotate(rows(t["wq"]), table, first).reshape(n, -1), k, v]
