"""The work this framework is measured by: prompt passes and decoding of its model shapes (lumen_amd.synth), and single products
through the C ABI.  Weights, tokens and operands are random; `exact` restates the models in float64 torch.

A model serves one live sequence after another, as in a program that answers: it is made once per process, with weights of a fixed
seed, and the states of a case bring new tokens to it (behind the same conversation, where there is one so far).  Passes of one case
go with states of that case only.

kind "matmul"   lumen_matmul_f32 / lumen_gemm_bf16w on the caller's buffers
     "prompt"   a prompt (or the new tokens of a turn, behind `past` cached ones) through a Llama; logits of the last token
     "decode"   `n` greedy tokens behind `past` cached ones, then the step whose logits a sampler would read
     "turn"     a layered hybrid model from its start: a prompt of `s` tokens, then `n` greedy tokens and one step more
"""
import math
import zlib

import numpy as np
import torch

from lumen_amd import synth
from lumen_amd._lib import check, lib
from lumen_amd.autograd import default_ctx
from lumen_amd.hybrid import HybridConfig, HybridLayer, HybridModel
from lumen_amd.models import LlamaModel

WEIGHT_SEED = 5
# Llama shapes of lumen_amd.synth; the wide one with 8 of its 32 layers (they are alike, and it is quicker to make)
LLAMA = {"tinyllama": dict(synth.TINYLLAMA_1B_LONG), "qwen3": dict(synth.QWEN3_0P6B), "llama2-7b": dict(synth.LLAMA2_7B, num_hidden_layers=8)}


def listed():
    return [
        # the smallest call there is: one row through a key projection; launch and host path
        {"name": "matmul 1x256x2048", "kind": "matmul", "m": 1, "n": 256, "k": 2048, "dtype": "f32"},
        # a projection of a prompt of a few hundred tokens as an operator of its own, sizes that fit no tile
        {"name": "matmul 301x4099x2052", "kind": "matmul", "m": 301, "n": 4099, "k": 2052, "dtype": "f32"},
        # answering: the headline shape behind a short prompt, and behind a cache that is nearly full
        {"name": "decode tinyllama 128", "kind": "decode", "model": "tinyllama", "past": 128, "n": 16},
        {"name": "decode tinyllama 3970", "kind": "decode", "model": "tinyllama", "past": 3970, "n": 8},
        # narrow layers, q / k norms, a head of a quarter of the weights
        {"name": "decode qwen3 261", "kind": "decode", "model": "qwen3", "past": 261, "n": 16},
        # wide layers, weights stored as bf16
        {"name": "decode llama2-7b 517", "kind": "decode", "model": "llama2-7b", "past": 517, "n": 8},
        # the new tokens of a chat turn behind the conversation so far
        {"name": "prompt tinyllama 301+23", "kind": "prompt", "model": "tinyllama", "past": 301, "s": 23},
        # a question, a document
        {"name": "prompt tinyllama 128", "kind": "prompt", "model": "tinyllama", "past": 0, "s": 128},
        {"name": "prompt tinyllama 3968", "kind": "prompt", "model": "tinyllama", "past": 0, "s": 3968},
        {"name": "prompt llama2-7b 509", "kind": "prompt", "model": "llama2-7b", "past": 0, "s": 509},
        # the hybrid designs: a long prompt through windows and recurrences; a short answer through experts and a matrix memory
        {"name": "turn pinavik 2048+0", "kind": "turn", "model": "pinavik", "width": 2048, "dtype": "bf16", "s": 2048, "n": 0},
        {"name": "turn nufapel 61+16", "kind": "turn", "model": "nufapel", "width": 2048, "dtype": "bf16", "s": 61, "n": 16},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matmul", "prompt", "prompt", "decode", "turn"])
    if kind == "matmul":
        # rows from one token to a long prompt, columns and depth over the shapes' projections; rows of whole 16-byte pieces
        return {"kind": kind, "m": _log_int(rng, 1, 4096), "n": _log_int(rng, 256, 11264), "k": _log_int(rng, 256, 11008) // 8 * 8,
                "dtype": rng.choice(["f32", "f32", "bf16"])}
    if kind == "turn":
        model = rng.choice(["pinavik", "nufapel"])
        return {"kind": kind, "model": model, "width": rng.choice([1024, 2048]), "dtype": rng.choice(["f32", "bf16"]),
                "s": _log_int(rng, 1, 2000), "n": rng.choice([0, 4, 16])}
    model = rng.choice(sorted(LLAMA))
    room = LLAMA[model]["max_seq_len"]
    if kind == "decode":
        return {"kind": kind, "model": model, "past": _log_int(rng, 16, room - 40), "n": rng.choice([1, 4, 12])}
    s = _log_int(rng, 2, room - 140)
    return {"kind": kind, "model": model, "past": rng.choice([0, 0, rng.randrange(1, min(1000, room - s))]), "s": s}


# ---------------------------------------------------------------------------------------------------- values
class Values:
    """Normal values for tensors by name: slices of one pool made from the seed, whose length is prime, so that a tensor longer than
    the pool repeats no row.  With bf16 every value of a matrix is one that bf16 holds."""
    POOL = 67108859

    def __init__(self, seed, bf16):
        g = torch.Generator("cuda").manual_seed(seed)
        self.pool = torch.randn(self.POOL, generator=g, device="cuda")
        self.seed, self.bf16, self.host = seed, bf16, {}

    def _pieces(self, name, n):
        at = (zlib.crc32(name.encode()) * 2654435761 + 97 * self.seed) % self.POOL
        if n <= self.POOL:
            at %= self.POOL - n + 1
        out = []
        while n > 0:
            take = min(n, self.POOL - at)
            out.append((at, at + take))
            n, at = n - take, 0
        return out

    def matrix(self, name, shape, std):
        """On the GPU, float32."""
        n = int(np.prod(shape))
        t = torch.cat([self.pool[a:b] for a, b in self._pieces(name, n)]) * std
        return (t.bfloat16().float() if self.bf16 else t).reshape(shape)

    def upload_form(self, name, shape, std):
        """The same values on the host: float32, or bf16 bits."""
        key = std
        if key not in self.host:
            t = self.pool * std
            self.host[key] = t.bfloat16().view(torch.int16).cpu().numpy().view(np.uint16) if self.bf16 else t.cpu().numpy()
        parts = [self.host[key][a:b] for a, b in self._pieces(name, int(np.prod(shape)))]
        return (parts[0] if len(parts) == 1 else np.concatenate(parts)).reshape(shape)

    def vector(self, name, shape):
        g = np.random.Generator(np.random.PCG64([self.seed, zlib.crc32(name.encode())]))
        return g.standard_normal(shape, dtype=np.float32)


def _tokens(seed, n, vocab, what):
    return np.random.Generator(np.random.PCG64([seed, zlib.crc32(what.encode())])).integers(0, vocab, n)


# ---------------------------------------------------------------------------------------------------- Llama
def _llama_shapes(c):
    H, I, V = c["hidden_size"], c["intermediate_size"], c["vocab_size"]
    D = c.get("head_dim") or H // c["num_attention_heads"]
    q, kv = c["num_attention_heads"] * D, c["num_key_value_heads"] * D
    yield "model.embed_tokens.weight", (V, H)
    for i in range(c["num_hidden_layers"]):
        p = "model.layers.%d." % i
        for n, s in (("self_attn.q_proj", (q, H)), ("self_attn.k_proj", (kv, H)), ("self_attn.v_proj", (kv, H)), ("self_attn.o_proj", (H, q)),
                     ("mlp.gate_proj", (I, H)), ("mlp.up_proj", (I, H)), ("mlp.down_proj", (H, I)),
                     ("input_layernorm", (H,)), ("post_attention_layernorm", (H,))):
            yield p + n + ".weight", s
        if c.get("qk_norm"):
            yield p + "self_attn.q_norm.weight", (D,)
            yield p + "self_attn.k_norm.weight", (D,)
    yield "model.norm.weight", (H,)
    if not c.get("tie_embeddings"):
        yield "lm_head.weight", (V, H)


def _gain(values, name, shape):
    return 1 + np.float32(0.1) * values.vector(name, shape)


def _llama_inputs(case, seed):
    c = LLAMA[case["model"]]
    n = case.get("s", 1)
    return _tokens(WEIGHT_SEED, case["past"], c["vocab_size"], "past"), _tokens(seed, n, c["vocab_size"], "new")


_models = {}


def _llama(name):
    if name not in _models:
        c = LLAMA[name]
        values = Values(WEIGHT_SEED, c.get("weight_dtype") == "bf16")
        model = LlamaModel(c)
        for n, shape in _llama_shapes(c):
            model.set_param(n, values.upload_form(n, shape, 0.02) if len(shape) == 2 else _gain(values, n, shape))
        _models[name] = model
    return _models[name]


def _prepare_llama(case, seed):
    model = _llama(case["model"])
    past, new = _llama_inputs(case, seed)
    if len(past):  # the conversation so far
        model.reset()
        model.forward(past, all_rows=False)
    return {"model": model, "past": len(past), "new": new, "n": case.get("n")}


def _run_prompt(s):
    s["model"].set_kv_len(s["past"])
    return s["model"].forward(s["new"], all_rows=False)


def _run_decode(s):
    m = s["model"]
    m.set_kv_len(s["past"])
    ids = m.decode_greedy(int(s["new"][0]), s["n"])
    return {"ids": ids, "logits": m.forward(ids[-1:], all_rows=False)}


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _exact_llama(case, seed):
    c = LLAMA[case["model"]]
    values = Values(WEIGHT_SEED, c.get("weight_dtype") == "bf16")
    P = {n: (values.matrix(n, s, 0.02).double() if len(s) == 2 else torch.from_numpy(_gain(values, n, s)).double().cuda()) for n, s in _llama_shapes(c)}
    head = P["model.embed_tokens.weight" if c.get("tie_embeddings") else "lm_head.weight"]
    H, Hq, Hkv, eps, L = c["hidden_size"], c["num_attention_heads"], c["num_key_value_heads"], c["rms_norm_eps"], c["num_hidden_layers"]
    D = c.get("head_dim") or H // Hq
    # the model's rotation angles are float32 products of a position and a float32 frequency
    freq = np.float32(1) / np.power(c["rope_theta"], np.arange(0, D, 2) / D).astype(np.float32)
    angle = torch.from_numpy((np.arange(c["max_seq_len"], dtype=np.float32)[:, None] * freq[None]).astype(np.float64)).cuda()
    cos, sin = torch.cos(angle), torch.sin(angle)
    cache = [None] * L

    def rotate(x, at):  # [T, heads, D]
        a, b = x[..., :D // 2], x[..., D // 2:]
        co, si = cos[at:at + len(x), None], sin[at:at + len(x), None]
        return torch.cat([a * co - b * si, b * co + a * si], -1)

    def forward(ids, at):
        x = P["model.embed_tokens.weight"][torch.as_tensor(np.asarray(ids, np.int64)).cuda()]
        T = len(ids)
        for i in range(L):
            w = lambda n: P["model.layers.%d.%s.weight" % (i, n)]  # noqa: E731
            h = _rms(x, eps) * w("input_layernorm")
            q, k, v = ((h @ w("self_attn.%s_proj" % n).T).reshape(T, -1, D) for n in "qkv")
            if c.get("qk_norm"):
                q, k = _rms(q, eps) * w("self_attn.q_norm"), _rms(k, eps) * w("self_attn.k_norm")
            q, k = rotate(q, at), rotate(k, at)
            if at:
                k, v = torch.cat([cache[i][0], k]), torch.cat([cache[i][1], v])
            cache[i] = (k, v)
            o = torch.empty_like(q)
            hidden = torch.arange(at + T, device="cuda")[None] > at + torch.arange(T, device="cuda")[:, None]
            for g in range(Hq):
                s = (q[:, g] @ k[:, g * Hkv // Hq].T.contiguous()) * D ** -0.5
                o[:, g] = torch.softmax(s.masked_fill(hidden, -math.inf), -1) @ v[:, g * Hkv // Hq].contiguous()
            x = x + o.reshape(T, -1) @ w("self_attn.o_proj").T
            h = _rms(x, eps) * w("post_attention_layernorm")
            x = x + (torch.nn.functional.silu(h @ w("mlp.gate_proj").T) * (h @ w("mlp.up_proj").T)) @ w("mlp.down_proj").T
        return (head @ (_rms(x[-1], eps) * P["model.norm.weight"])).cpu().numpy()

    past, new = _llama_inputs(case, seed)
    if len(past):
        forward(past, 0)
    if case["kind"] == "prompt":
        return forward(new, len(past))
    tok, at = int(new[0]), len(past)
    for _ in range(case["n"]):
        tok, at = int(np.argmax(forward([tok], at))), at + 1
    return {"ids": None, "logits": forward([tok], at)}


# ---------------------------------------------------------------------------------------------------- hybrid designs
def _design(case):
    """(fields of the configuration, layers) of the shapes that bench.py times."""
    W = case["width"]
    room = 4096
    if case["model"] == "pinavik":
        delta = dict(mixer="channel_delta", heads=W // 128, kv_heads=W // 128, dim=128, vdim=128, conv=4, rank_lo=128, rank_hi=128, ff=4 * W)
        group = [dict(mixer="attention", heads=W // 64, kv_heads=W // 256, dim=64, vdim=64, window=1024, scale=0.125, softcap=30.0, ff=4 * W),
                 delta, dict(mixer="wkv", heads=W // 64, kv_heads=W // 64, dim=64, vdim=64, rank_lo=64, ff=4 * W), delta]
        return dict(embed_scale=W ** 0.5, norm_offset=1.0, residual_mult=0.6, max_seq_len=room), group * 3
    moe = dict(ff=W // 4, ff_kind="experts", experts=32, top=8, groups=8, keep=4, router_scale=1.0, limit=7.0)
    par = dict(mixer="parallel", heads=W // 64, kv_heads=W // 256, dim=64, vdim=64, scale=0.125, bias_rows=32, bias_max=128,
               mem_heads=W // 256, mem_dim=128, mem_vdim=128, gate_cap=15.0)
    gen = dict(mixer="general_delta", heads=W // 64, kv_heads=W // 64, dim=64, vdim=64, rank_lo=64)
    layers = [dict(gen if i % 2 else par, **(moe if i else dict(ff=4 * W, ff_kind="gelu"))) for i in range(12)]
    return dict(max_seq_len=room, norm_kind="dyt", loop_kind="add", residual_gate=True, max_positions=room, logit_softcap=30.0), layers


HYBRID_VOCAB, LOOP, EPS = 32000, (4, 8, 2), 1e-6


def _hybrid_shapes(case):
    W, V = case["width"], HYBRID_VOCAB
    top, layers = _design(case)
    nufapel = case["model"] == "nufapel"

    def norm(n):
        return {n: (W,), n + ".b": (W,), n + ".alpha": ()} if nufapel else {n: (W,)}
    s = dict({"embed": (V, W), "head": (V, W), "loop.step": (LOOP[2], W)}, **norm("final.norm"))
    s.update({"pos": (top["max_positions"], W)} if nufapel else {"loop.in": (W, 2 * W)})
    for i, y in enumerate(layers):
        p, H, G, D, Dv = "l%d." % i, y["heads"], y["kv_heads"], y["dim"], y["vdim"]
        n, x = H * D, p + "mix."
        s.update(norm(p + "norm1"))
        s.update(norm(p + "norm2"))
        if nufapel:
            s.update({p + "rg1": (W, W), p + "rg1.b": (W,), p + "rg2": (W, W), p + "rg2.b": (W,)})
        if y["mixer"] == "attention":
            s.update({x + "q": (n, W), x + "k": (G * D, W), x + "v": (G * Dv, W), x + "g": (H * Dv, W), x + "o": (W, H * Dv),
                      x + "q.norm": (n,), x + "k.norm": (G * D,), x + "r1": (H,), x + "r2": (H,)})
        elif y["mixer"] == "wkv":
            s.update({x + k: (n, W) for k in "rkvg"})
            s.update({x + "mu." + k: (W,) for k in "rkvgw"})
            s.update({x + "w1": (y["rank_lo"], W), x + "w2": (n, y["rank_lo"]), x + "w0": (n,), x + "u": (H, D), x + "norm": (n,), x + "o": (W, n)})
        elif y["mixer"] == "channel_delta":
            lo, hi, t = y["rank_lo"], y["rank_hi"], y["conv"]
            s.update({x + "q": (G * D, W), x + "k": (G * D, W), x + "v": (H * Dv, W), x + "q.conv": (G * D, t), x + "k.conv": (G * D, t),
                      x + "v.conv": (H * Dv, t), x + "b": (H, W), x + "A_log": (H,), x + "norm": (Dv,), x + "a1": (lo, W), x + "a2": (n, lo),
                      x + "dt_bias": (n,), x + "g1": (hi, W), x + "g2": (H * Dv, hi), x + "o": (W, H * Dv)})
        elif y["mixer"] == "general_delta":
            s.update({x + k: (n, W) for k in "rkvga"})
            s.update({x + "a.b": (n,), x + "w1": (y["rank_lo"], W), x + "w2": (n, y["rank_lo"]), x + "w0": (n,), x + "norm": (n,), x + "o": (W, n)})
        else:
            a, r, Hm, nm, nv = x + "left.", x + "right.", y["mem_heads"], y["mem_heads"] * y["mem_dim"], y["mem_heads"] * y["mem_vdim"]
            s.update({a + "q": (n, W), a + "k": (G * D, W), a + "v": (G * Dv, W), a + "rel": (y["bias_rows"], H), a + "temp": (H,), a + "sink": (H,),
                      a + "g": (H, W), a + "o": (W, H * Dv), a + "out": (W,), r + "q": (nm, W), r + "k": (nm, W), r + "v": (nv, W), r + "g": (nv, W),
                      r + "o": (W, nv), r + "norm": (nv,), r + "i": (Hm, W), r + "i.b": (Hm,), r + "f": (Hm, W), r + "f.b": (Hm,), r + "out": (W,)})
        F, kind = y["ff"], y.get("ff_kind", "polynorm")
        if kind == "experts":
            s[p + "mlp.router"] = (y["experts"], W)
            for e in range(y["experts"]):
                s.update({p + "mlp.e%d.gate" % e: (F, W), p + "mlp.e%d.up" % e: (F, W), p + "mlp.e%d.down" % e: (W, F)})
        else:
            s.update({p + "mlp.up": (F, W), p + "mlp.down": (W, F)})
            if kind == "polynorm":
                s[p + "mlp.act"] = (4,)
    return s


def _hybrid_std(name, shape, nufapel):
    """Scale of a large matrix; None for a small tensor with a rule of its own."""
    leaf = name.split(".")[-1]
    if len(shape) != 2 or leaf in ("u", "conv", "step", "rel"):
        return None
    if leaf == "pos":
        return 0.3
    if nufapel and leaf == "embed":
        return 1.0
    return shape[1] ** -0.5 * (2.0 if nufapel and name.endswith(("mlp.router", "head", "left.q")) else 1.0)


def _hybrid_small(values, name, shape, nufapel):
    a, leaf, f = values.vector(name, shape), name.split(".")[-1], np.float32
    if nufapel:
        if leaf == "alpha":
            return np.asarray(f(0.6) + f(0.1) * a, f)
        if name.endswith(".f.b"):
            return 3 + a
        if (name.endswith(".b") and "norm" in name) or name == "loop.step":
            return a * f(0.3)
        return 1 + a * f(0.2) if leaf in ("norm1", "norm2", "norm", "out", "temp") else a
    if name.endswith("conv"):
        return a * f(shape[-1] ** -0.5)
    if leaf in ("norm1", "norm2") or name in ("final.norm", "loop.step"):
        return a * f(0.1)
    if leaf == "norm":
        return 1 + a * f(0.1)
    if leaf == "act":
        return np.array([0.5, 0.3, 0.2, 0.05], f) + a * f(0.02)
    if leaf in ("r1", "r2") or ".mu." in name:
        return np.abs(a) * f(0.3)
    return a * f(0.5) - f(2.5) if leaf in ("w0", "dt_bias") else a * f(0.3)


def _hybrid(case):
    key = (case["model"], case["width"], case["dtype"])
    if key not in _models:
        top, layers = _design(case)
        nufapel = case["model"] == "nufapel"
        values = Values(WEIGHT_SEED, case["dtype"] == "bf16")
        model = HybridModel(HybridConfig(HYBRID_VOCAB, case["width"], [HybridLayer(**y) for y in layers], *LOOP, norm_eps=EPS,
                                         weight_dtype=case["dtype"], **top))
        for name, shape in _hybrid_shapes(case).items():
            std = _hybrid_std(name, shape, nufapel)
            model.set_param(name, _hybrid_small(values, name, shape, nufapel) if std is None else values.upload_form(name, shape, std))
        _models[key] = model
    return _models[key]


def _prepare_turn(case, seed):
    return {"model": _hybrid(case), "new": _tokens(seed, case["s"], HYBRID_VOCAB, "new"), "n": case["n"]}


def _run_turn(s):
    m = s["model"]
    m.reset()
    last = m.step(s["new"], [len(s["new"]) - 1])[0]
    if not s["n"]:
        return {"logits": last}
    ids = m.decode_greedy(int(np.argmax(last)), s["n"])
    return {"logits": last, "ids": ids, "next": m.step(ids[-1:], [0])[0]}


def _exact_turn(case, seed):
    nufapel = case["model"] == "nufapel"
    if nufapel and case["s"] + case["n"] > 96:
        return None  # thousands of choices of experts, some of them so close that 32 bits may decide them either way
    top, layers = _design(case)
    values, W = Values(WEIGHT_SEED, case["dtype"] == "bf16"), case["width"]
    shapes = _hybrid_shapes(case)

    def P(name):
        std = _hybrid_std(name, shapes[name], nufapel)
        return (torch.from_numpy(np.asarray(_hybrid_small(values, name, shapes[name], nufapel))).cuda() if std is None else
                values.matrix(name, shapes[name], std)).double()

    def norm(x, n):
        if nufapel:
            return torch.tanh(P(n + ".alpha") * x) * P(n) + P(n + ".b")
        return _rms(x, EPS) * (1 + P(n))

    def shift(h):
        return torch.cat([torch.zeros_like(h[:1]), h[:-1]])

    def attend(q, k, v, score):  # score(s, distance, head)
        T, Hq = q.shape[0], q.shape[1]
        o = q.new_empty(T, Hq, v.shape[2])
        dist = (torch.arange(T, device="cuda")[:, None] - torch.arange(T, device="cuda")[None]).double()
        for g in range(Hq):
            j = g * k.shape[1] // Hq
            s, extra = score(q[:, g] @ k[:, j].T.contiguous(), dist, g)
            s = torch.cat([s.masked_fill(dist < 0, -math.inf), extra], 1)
            o[:, g] = torch.softmax(s, -1)[:, :T] @ v[:, j].contiguous()
        return o

    def mixer(i, y, h):
        T, H, G, D, Dv, p = len(h), y["heads"], y["kv_heads"], y["dim"], y["vdim"], "l%d.mix." % i
        proj = lambda n, *sh: (h @ P(p + n).T).reshape(T, *sh)  # noqa: E731
        if y["mixer"] == "attention":
            q = (_rms(proj("q", H * D), EPS) * P(p + "q.norm")).reshape(T, H, D)
            k = (_rms(proj("k", G * D), EPS) * P(p + "k.norm")).reshape(T, G, D)
            r1, r2, cap = P(p + "r1"), P(p + "r2"), y["softcap"]

            def score(s, d, g):
                s = cap * torch.tanh(s * y["scale"] / cap) - r1[g] * torch.log1p(r2[g] * d.clamp(min=0))
                return s.masked_fill(d >= y["window"], -math.inf), s[:, :0]
            o = attend(q, k, proj("v", G, Dv), score).reshape(T, -1) * torch.sigmoid(proj("g", H * Dv))
            return o @ P(p + "o").T
        if y["mixer"] == "wkv":
            m = {n: h + (shift(h) - h) * P(p + "mu." + n) for n in "rkvgw"}
            r, k, v = ((m[n] @ P(p + n).T).reshape(T, H, D) for n in "rkv")
            w = torch.exp(-torch.exp(torch.tanh(m["w"] @ P(p + "w1").T) @ P(p + "w2").T + P(p + "w0"))).reshape(T, H, D)
            u, S, o = P(p + "u")[:, :, None], h.new_zeros(H, D, D), torch.empty_like(v)
            for t in range(T):
                kv = k[t, :, :, None] * v[t, :, None]
                o[t] = (r[t, :, :, None] * (S + u * kv)).sum(1)
                S = w[t, :, :, None] * S + kv
            return (_rms(o, EPS).reshape(T, -1) * P(p + "norm") * torch.nn.functional.silu(m["g"] @ P(p + "g").T)) @ P(p + "o").T
        if y["mixer"] == "channel_delta":
            def conv(n):
                x, taps = h @ P(p + n).T, P(p + n + ".conv")
                out, back = taps[:, -1] * x, x
                for j in range(2, taps.shape[1] + 1):
                    back = shift(back)
                    out = out + taps[:, -j] * back
                return torch.nn.functional.silu(out)
            unit = lambda x: x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
            q, k, v = unit(conv("q").reshape(T, G, D)) * D ** -0.5, unit(conv("k").reshape(T, G, D)), conv("v").reshape(T, H, Dv)
            beta = torch.sigmoid(proj("b", H))
            z = torch.nn.functional.softplus((h @ P(p + "a1").T) @ P(p + "a2").T + P(p + "dt_bias"), threshold=1e9).reshape(T, H, D)
            w = torch.exp(-torch.exp(P(p + "A_log"))[:, None] * z)
            S, o = h.new_zeros(H, D, Dv), torch.empty_like(v)
            for t in range(T):
                S = w[t, :, :, None] * S
                S = S + k[t, :, :, None] * (beta[t, :, None] * (v[t] - (S * k[t, :, :, None]).sum(1)))[:, None]
                o[t] = (S * q[t, :, :, None]).sum(1)
            return ((_rms(o, EPS) * P(p + "norm")).reshape(T, -1) * torch.sigmoid((h @ P(p + "g1").T) @ P(p + "g2").T)) @ P(p + "o").T
        if y["mixer"] == "general_delta":
            r, k, v = (proj(n, H, D) for n in "rkv")
            w = torch.exp(-math.exp(-0.5) * torch.sigmoid(torch.tanh(h @ P(p + "w1").T) @ P(p + "w2").T + P(p + "w0"))).reshape(T, H, D)
            a = torch.sigmoid(proj("a", H * D) + P(p + "a.b")).reshape(T, H, D)
            u = k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)
            S, o = h.new_zeros(H, D, D), torch.empty_like(v)
            for t in range(T):
                seen = (u[t, :, :, None] * S).sum(1)
                S = w[t, :, :, None] * S - (a[t] * u[t])[:, :, None] * seen[:, None] + k[t, :, :, None] * v[t, :, None]
                o[t] = (S * r[t, :, :, None]).sum(1)
            return (_rms(o, EPS).reshape(T, -1) * P(p + "norm") * torch.sigmoid(proj("g", H * D))) @ P(p + "o").T
        rows, most = y["bias_rows"], y["bias_max"]
        half = rows // 2
        far = lambda n: n if n < half else min(rows - 1, half + int(math.floor(math.log(n / half) / math.log(most / half) * (rows - half) + 1e-9)))  # noqa: E731
        bucket = torch.tensor([far(n) for n in range(T)], device="cuda")
        rel, temp, sink = P(p + "left.rel"), P(p + "left.temp"), P(p + "left.sink")

        def score(s, d, g):
            return s * y["scale"] * temp[g] + rel[bucket[d.clamp(min=0).long()], g], sink[g].expand(T, 1)
        o = attend(proj("left.q", H, D), proj("left.k", G, D), proj("left.v", G, Dv), score) * torch.sigmoid(proj("left.g", H))[:, :, None]
        left = o.reshape(T, -1) @ P(p + "left.o").T
        Hm, Dm, Vm, cap = y["mem_heads"], y["mem_dim"], y["mem_vdim"], y["gate_cap"]
        q, k, v = proj("right.q", Hm, Dm) * Dm ** -0.5, proj("right.k", Hm, Dm), proj("right.v", Hm, Vm)
        gi = cap * torch.tanh((proj("right.i", Hm) + P(p + "right.i.b")) / cap)
        gf = torch.nn.functional.logsigmoid(cap * torch.tanh((proj("right.f", Hm) + P(p + "right.f.b")) / cap))
        S, n, m, o = h.new_zeros(Hm, Dm, Vm), h.new_zeros(Hm, Dm), h.new_zeros(Hm), torch.empty_like(v)
        for t in range(T):
            new = torch.maximum(gf[t] + m, gi[t])
            keep, add, m = torch.exp(gf[t] + m - new), torch.exp(gi[t] - new), new
            S = keep[:, None, None] * S + add[:, None, None] * k[t, :, :, None] * v[t, :, None]
            n = keep[:, None] * n + add[:, None] * k[t]
            o[t] = (S * q[t, :, :, None]).sum(1) / (torch.maximum((n * q[t]).sum(1).abs(), torch.exp(-m)) + 1e-6)[:, None]
        right = (_rms(o, EPS).reshape(T, -1) * P(p + "right.norm") * torch.sigmoid(proj("right.g", Hm * Vm))) @ P(p + "right.o").T
        return 0.5 * (_rms(left, EPS) * P(p + "left.out") + _rms(right, EPS) * P(p + "right.out"))

    def feed_forward(i, y, h):
        p, kind = "l%d.mlp." % i, y.get("ff_kind", "polynorm")
        if kind == "gelu":
            z = h @ P(p + "up").T
            return (0.5 * z * (1 + torch.erf(z / math.sqrt(2.0)))) @ P(p + "down").T
        if kind == "polynorm":
            z, c = h @ P(p + "up").T, P(p + "act")
            return (c[0] * _rms(z, EPS) + c[1] * _rms(z ** 2, EPS) + c[2] * _rms(z ** 3, EPS) + c[3]) @ P(p + "down").T
        T, E, g = len(h), y["experts"], y["groups"]
        s = torch.sigmoid(h @ P(p + "router").T)
        best = s.reshape(T, g, E // g).topk(2, -1).values.sum(-1).topk(y["keep"], -1).indices
        open_ = torch.zeros(T, g, device="cuda", dtype=torch.bool).scatter_(1, best, True).repeat_interleave(E // g, 1)
        w, at = s.masked_fill(~open_, -1.0).topk(y["top"], -1)
        weight = torch.zeros_like(s).scatter_(1, at, w / w.sum(-1, keepdim=True) * y["router_scale"])
        out = torch.zeros_like(h)
        for e in range(E):
            a = (h @ P(p + "e%d.gate" % e).T).clamp(max=y["limit"])
            b = (h @ P(p + "e%d.up" % e).T).clamp(-y["limit"], y["limit"])
            out += weight[:, e:e + 1] * ((a * torch.sigmoid(1.702 * a) * (b + 1)) @ P(p + "e%d.down" % e).T)
        return out

    def forward(ids):  # the whole sequence from its start; logits of the last token
        ids = torch.as_tensor(np.asarray(ids, np.int64)).cuda()
        x = x0 = P("embed")[ids] * top.get("embed_scale", 1.0) + (P("pos")[:len(ids)] if nufapel else 0)
        a, b, times = LOOP
        runs = [(i, None) for i in range(a)] + [(i, t if i == a else None) for t in range(times) for i in range(a, b)]
        for i, t in runs + [(i, None) for i in range(b, len(layers))]:
            if t is not None:
                x = (x if nufapel else torch.cat([x, x0], 1) @ P("loop.in").T) + P("loop.step")[t]
            for k, part in ((1, mixer), (2, feed_forward)):
                h = norm(x, "l%d.norm%d" % (i, k))
                gate = torch.sigmoid(h @ P("l%d.rg%d" % (i, k)).T + P("l%d.rg%d.b" % (i, k))) if nufapel else top["residual_mult"]
                x = x + part(i, layers[i], h) * gate
        z = norm(x[-1:], "final.norm")[0] @ P("head").T
        return (30.0 * torch.tanh(z / 30.0) if nufapel else z).cpu().numpy()

    ids = list(_tokens(seed, case["s"], HYBRID_VOCAB, "new"))
    last = forward(ids)
    if not case["n"]:
        return {"logits": last}
    if case["s"] > 96:
        return {"logits": last, "ids": None, "next": None}  # the whole sequence once more for every token
    tok = int(np.argmax(last))
    for _ in range(case["n"]):
        ids.append(tok)
        tok = int(np.argmax(forward(ids)))
    return {"logits": last, "ids": None, "next": forward(ids + [tok])}


# ---------------------------------------------------------------------------------------------------- single products
def _matmul_inputs(case, seed):
    values = Values(seed, case["dtype"] == "bf16")
    a = torch.randn(case["m"], case["k"], generator=torch.Generator("cuda").manual_seed(seed + 1), device="cuda")
    return a, values.matrix("w", (case["n"], case["k"]), 0.02)


def _prepare_matmul(case, seed):
    a, w = _matmul_inputs(case, seed)
    if case["dtype"] == "bf16":
        w = w.bfloat16()
    c = torch.empty(case["m"], case["n"], device="cuda")
    torch.cuda.synchronize()  # the library works on a stream of its own
    return dict(case, ctx=default_ctx().handle, a=a, w=w, c=c)


def _run_matmul(s):
    a, w, c = s["a"].data_ptr(), s["w"].data_ptr(), s["c"].data_ptr()
    if s["dtype"] == "f32":
        check(lib.lumen_matmul_f32(s["ctx"], a, w, c, s["m"], s["n"], s["k"], s["k"]))
    elif s["m"] == 1:
        check(lib.lumen_gemv_bf16w(s["ctx"], w, a, c, s["n"], s["k"]))
    else:
        check(lib.lumen_gemm_bf16w(s["ctx"], a, w, c, s["m"], s["n"], s["k"]))
    return s["c"]


def _exact_matmul(case, seed):
    a, w = _matmul_inputs(case, seed)
    return a.double() @ w.double().T


# ---------------------------------------------------------------------------------------------------- the interface
_PREPARE = {"matmul": _prepare_matmul, "prompt": _prepare_llama, "decode": _prepare_llama, "turn": _prepare_turn}
_RUN = {"matmul": _run_matmul, "prompt": _run_prompt, "decode": _run_decode, "turn": _run_turn}
_EXACT = {"matmul": _exact_matmul, "prompt": _exact_llama, "decode": _exact_llama, "turn": _exact_turn}


def prepare(case, seed):
    return dict(_PREPARE[case["kind"]](case, seed), kind=case["kind"])


def run(state):
    return _RUN[state["kind"]](state)


def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)


def work(case):
    """Weights of the layers once per pass over them (per decoded token), caches' rows once, 2 operations per weight and token."""
    if case["kind"] == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 4 * (m * k + m * n) + n * k * (4 if case["dtype"] == "f32" else 2), "flops": 2 * m * n * k}
    if case["kind"] == "turn":
        return _work_turn(case)
    c = LLAMA[case["model"]]
    L, D = c["num_hidden_layers"], c.get("head_dim") or c["hidden_size"] // c["num_attention_heads"]
    inner = sum(int(np.prod(s)) for n, s in _llama_shapes(c) if len(s) == 2 and ".layers." in n)
    head, size = c["vocab_size"] * c["hidden_size"], 2 if c.get("weight_dtype") == "bf16" else 4
    row = 2 * L * c["num_key_value_heads"] * D * 4  # keys and values of a token
    score = 4 * L * c["num_attention_heads"] * D    # operations per token and key it sees
    if case["kind"] == "decode":
        steps = case["n"] + 1
        keys = steps * case["past"] + steps * (steps + 1) // 2
        return {"bytes": steps * size * (inner + head) + row * keys, "flops": 2 * steps * (inner + head) + score * keys}
    s, past = case["s"], case["past"]
    return {"bytes": size * (inner + head) + row * (past + s) + s * c["hidden_size"] * 4,
            "flops": 2 * (s * inner + head) + score * (s * past + s * (s + 1) // 2)}


def _work_turn(case):
    shapes, (top, layers), size = _hybrid_shapes(case), _design(case), 2 if case["dtype"] == "bf16" else 4
    runs = list(range(LOOP[0])) + list(range(LOOP[0], LOOP[1])) * LOOP[2] + list(range(LOOP[1], len(layers)))
    head = case["width"] * HYBRID_VOCAB
    nbytes = flops = 0.0
    steps = case["n"] + 1 if case["n"] else 0
    for passes, tokens in ((1, case["s"]), (steps, 1)):  # the prompt, then single tokens
        for i in runs:
            y, dense, expert = layers[i], 0, 0
            for n, sh in shapes.items():
                if n.startswith("l%d." % i) and len(sh) == 2:
                    if ".mlp.e" in n:
                        expert += int(np.prod(sh))
                    else:
                        dense += int(np.prod(sh))
            used, touched = (y["top"] / y["experts"], min(1.0, tokens * y["top"] / y["experts"])) if expert else (0, 0)
            nbytes += passes * size * (dense + touched * expert)
            flops += passes * tokens * 2 * (dense + used * expert)
            state = y["heads"] * y["dim"] * y["vdim"] + y.get("mem_heads", 0) * y.get("mem_dim", 0) * y.get("mem_vdim", 0)
            if y["mixer"] in ("attention", "parallel"):
                seen = min(y.get("window") or case["s"], case["s"])
                keys = tokens * seen / 2 if tokens > 1 else seen
                flops += passes * 4 * keys * y["heads"] * y["dim"]
                nbytes += passes * 4 * y["kv_heads"] * (y["dim"] + y["vdim"]) * (tokens if tokens > 1 else seen)
                state = y.get("mem_heads", 0) * y.get("mem_dim", 0) * y.get("mem_vdim", 0)
            flops += passes * tokens * 6 * state
            nbytes += passes * 8 * state
        nbytes += passes * size * head
        flops += passes * 2 * head
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Four times what these passes were measured off the float64 restatements: products of 32-bit sums 3e-7, logits up to 1.6e-5 (16 and more
    sums of thousands of terms one after the other, over up to four thousand positions)."""
    if case["kind"] == "matmul":
        return {"rel": 1.5e-6}
    if case.get("model") == "nufapel" and case["s"] + case["n"] > 96:
        return {"rel": 1e-2, "max": 0.3}  # a token's eighth and ninth expert may be a tie to 32 bits: their outputs change places
    return {"rel": 6e-5}
