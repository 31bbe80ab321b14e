"""Performance cases of the framework: the calls a program that serves Gemma 3 makes, from one token of the
tiny model to a long prompt, each through a public entry point of gemma_hip.

A case is a dict of plain values:

  kind    "step"       runGemmaInferenceCached: one token at position `start`, logits to the host
          "generate"   gh.generate at position `start`: `tokens` prompt tokens fed one per step, then `new` ids
                       on the device, then one step whose logits come back
          "prefill"    gh.prefill of `tokens` prompt tokens at position `start`, last logits to the host
          "matvec"     gh_q4_0_matvec, rows x cols, on device vectors
          "attention"  gh_attention_decode: one query over cache rows [begin, end)
  model   a preset of the library; `layers` of it; `weights` "q4_0" (a GGUF file's) or "f32" (a SafeTensors
          checkpoint's)

Weights, prompts, caches and vectors come from the seed alone.  exact() restates the arithmetic in 64 bits with
plain torch.
"""
from __future__ import annotations

import ctypes
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "gemma.hs_amd"))
import gemma_hip as gh  # noqa: E402

# hidden, heads, kv heads, head_dim, ffn, vocab, window, global layer every, theta local / global, cache capacity
SHAPES = {
    "tiny": (128, 4, 1, 32, 512, 1024, 0, 0, 1e4, 1e4, 2048),
    "gemma3-1b": (1152, 4, 1, 256, 6912, 262144, 512, 6, 1e4, 1e6, 2048),
    "gemma3-4b": (2560, 8, 4, 256, 10240, 262144, 1024, 6, 1e4, 1e6, 8192),
}
EPS = 1e-6


def listed():
    def model(name, kind, which, layers, weights, start, tokens, new=0, temperature=0.0, top_k=0):
        return {"name": name, "kind": kind, "model": which, "layers": layers, "weights": weights, "start": start,
                "tokens": tokens, "new": new, "temperature": temperature, "top_k": top_k}

    return [
        # the smallest call there is: one token of the CPU-sized f32 model, all launches and latency
        model("tiny_step_f32", "step", "tiny", 2, "f32", 17, 1),
        # greedy decoding after a short prompt: what most generated tokens cost (the benchmark's positions)
        model("decode_1b", "generate", "gemma3-1b", 26, "q4_0", 128, 1, 48),
        # a host-driven chat loop: one sampled token (top-k, temperature) late in a long conversation
        model("step_1b_sampled", "step", "gemma3-1b", 26, "q4_0", 1500, 1, 0, 0.8, 40),
        # the larger model decoding behind a 4096-token context
        model("decode_4b_4096", "generate", "gemma3-4b", 34, "q4_0", 4096, 1, 16),
        # decoding an f32 checkpoint (one period of the 1B model's layers): four times the bytes a weight
        model("decode_f32", "generate", "gemma3-1b", 6, "f32", 200, 3, 16),
        # an ordinary prompt: the benchmark's 128 tokens
        model("prefill_1b_128", "prefill", "gemma3-1b", 26, "q4_0", 0, 128),
        # a document as the prompt: nearly the whole default cache, a ragged last pass
        model("prefill_1b_1907", "prefill", "gemma3-1b", 26, "q4_0", 0, 1907),
        # the second turn of a chat: a short odd prompt behind what is already cached
        model("prefill_1b_turn", "prefill", "gemma3-1b", 26, "q4_0", 611, 37),
        # a long prompt for the larger model (two periods of its layers)
        model("prefill_4b_1024", "prefill", "gemma3-4b", 12, "q4_0", 0, 1024),
        # a prompt for an f32 checkpoint
        model("prefill_f32_300", "prefill", "gemma3-1b", 6, "f32", 0, 300),
        # runLinearQ4 on a resident matrix, the largest there is: the 262144-row LM head
        {"name": "matvec_lm_head", "kind": "matvec", "rows": 262144, "cols": 1152, "softcap": False},
        # one query of the 1B model's global layers over an 8192-position cache
        {"name": "attention_8192", "kind": "attention", "heads": 4, "kv_heads": 1, "head_dim": 256, "begin": 0,
         "end": 8192},
    ]


def draw(rng):
    def log(a, b):
        return max(a, min(b, int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))))

    kind = rng.choice(["step", "generate", "generate", "prefill", "prefill", "prefill", "matvec", "attention"])
    if kind == "matvec":
        cols = 32 * log(16, 320)  # 512 .. 10240 columns
        return {"kind": kind, "rows": log(100, min(262144, 262144 * 1152 // cols)), "cols": cols,
                "softcap": rng.random() < 0.25}
    if kind == "attention":
        heads, kv_heads = rng.choice([(4, 1), (8, 4), (8, 8), (8, 2)])
        end = log(16, 32768 // kv_heads)
        begin = max(0, end - rng.choice([512, 1024])) if rng.random() < 0.4 else 0
        return {"kind": kind, "heads": heads, "kv_heads": kv_heads, "head_dim": 256, "begin": begin, "end": end}
    which, layers, weights = rng.choice([("tiny", 2, "f32"), ("gemma3-1b", 26, "q4_0"), ("gemma3-1b", 26, "q4_0"),
                                         ("gemma3-4b", 12, "q4_0"), ("gemma3-1b", 6, "f32")])
    c = {"kind": kind, "model": which, "layers": layers, "weights": weights, "new": 0, "temperature": 0.0, "top_k": 0}
    if kind == "prefill":
        most = {"tiny": 1900, "gemma3-1b": 1900, "gemma3-4b": 1000}[which] if weights == "q4_0" or which == "tiny" else 400
        c["tokens"] = log(2, most)
        c["start"] = rng.randrange(0, 1 + min(1000, 1950 - c["tokens"])) if rng.random() < 0.3 else 0
    else:
        c["start"] = log(8, 1900 if which != "gemma3-4b" else 6000)
        c["tokens"] = 1 if kind == "step" else log(1, 12)
        c["new"] = 0 if kind == "step" else log(2, 48 if layers == 26 else 32 if weights == "q4_0" else 16)
        if kind == "step" and rng.random() < 0.5:
            c["temperature"], c["top_k"] = 0.7, rng.choice([0, 40])
    return c


# ------------------------------------------------------------------ inputs
_ctx = []


def _context():
    """The program's one context."""
    if not _ctx:
        _ctx.append(gh.Context(0))
    return _ctx[0]


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(1_000_003 * int(seed) + 17)
    return g


def _q4_blocks(g, rows, cols):
    """GGUF Q4_0 blocks [rows, cols/32, 18] as a quantiser leaves them: codes bell-shaped around 8, scales of
    either sign."""
    nb = cols // 32
    q = torch.randn(rows, nb, 32, generator=g, device="cuda").mul_(2.7).add_(8.0).round_().clamp_(0, 15).to(torch.uint8)
    d = torch.rand(rows, nb, 1, generator=g, device="cuda").mul_(0.008).add_(0.006)
    d *= torch.where(torch.rand(rows, nb, 1, generator=g, device="cuda") < 0.5, -1.0, 1.0)
    return torch.cat([d.half().view(torch.uint8), q[..., :16] | (q[..., 16:] << 4)], dim=2)


def _q4_values(raw):
    """The 64-bit values (q - 8) * d of _q4_blocks."""
    rows, nb, _ = raw.shape
    d = raw[..., :2].contiguous().view(torch.float16).double()
    q = torch.cat([raw[..., 2:] & 15, raw[..., 2:] >> 4], dim=2).double()
    return ((q - 8.0) * d).reshape(rows, nb * 32)


def _tensors(case, g):
    """(name, is_matrix, values) of every tensor in a fixed order; matrices as Q4_0 blocks or f32 [rows, cols]."""
    H, nq, nkv, hd, F, V = SHAPES[case["model"]][:6]

    def mat(rows, cols):
        if case["weights"] == "q4_0":
            return _q4_blocks(g, rows, cols)
        return torch.randn(rows, cols, generator=g, device="cuda").mul_(0.02)

    def vec(n):
        return torch.randn(n, generator=g, device="cuda").mul_(0.1)

    yield "token_embd.weight", True, mat(V, H)
    yield "output_norm.weight", False, vec(H)
    for layer in range(case["layers"]):
        p = "blk.%d." % layer
        for name, rows, cols in (("attn_q", nq * hd, H), ("attn_k", nkv * hd, H), ("attn_v", nkv * hd, H),
                                 ("attn_output", H, nq * hd), ("ffn_gate", F, H), ("ffn_up", F, H), ("ffn_down", H, F)):
            yield p + name + ".weight", True, mat(rows, cols)
        for name, n in (("attn_norm", H), ("attn_q_norm", hd), ("attn_k_norm", hd), ("post_attention_norm", H),
                        ("ffn_norm", H), ("post_ffw_norm", H)):
            yield p + name + ".weight", False, vec(n)


def _tokens(case, seed):
    """Token ids of the cached context, of this pass, and of the closing step."""
    V = SHAPES[case["model"]][5]
    ids = np.random.default_rng([int(seed), 5]).integers(0, V, case["start"] + case["tokens"] + 1).astype(np.int32)
    return ids[:case["start"]], ids[case["start"]:-1], int(ids[-1])


def _attention_inputs(case, seed):
    g = _generator(seed)
    rows, hd = case["end"] * case["kv_heads"], case["head_dim"]
    q = torch.randn(case["heads"] * hd, generator=g, device="cuda")
    k = torch.randn(rows, hd, generator=g, device="cuda")
    v = torch.randn(rows, hd, generator=g, device="cuda")
    return q, k, v


def prepare(case, seed):
    ctx = _context()
    if case["kind"] == "matvec":
        g = _generator(seed)
        raw = _q4_blocks(g, case["rows"], case["cols"])
        w = gh.Q4Tensor(ctx, raw.cpu().numpy().reshape(-1), case["rows"], case["cols"])
        x = torch.randn(case["cols"], generator=g, device="cuda")
        return {"case": case, "w": w, "x": x, "y": torch.empty(case["rows"], device="cuda")}
    if case["kind"] == "attention":
        q, k, v = _attention_inputs(case, seed)
        return {"case": case, "q": q, "k": k, "v": v, "out": torch.empty_like(q)}
    cfg = gh.preset(case["model"])
    cfg.n_layers = case["layers"]
    model = gh.GemmaModel(ctx, cfg)
    for name, is_matrix, t in _tensors(case, _generator(seed)):
        q4 = is_matrix and case["weights"] == "q4_0"
        model.set_tensor(name, t.cpu().numpy().reshape(-1), gh.DTYPE_Q4_0 if q4 else gh.DTYPE_F32)
    cache = gh.KVCache(model, SHAPES[case["model"]][10])
    if case["temperature"] > 0:
        cache.set_sampling(case["temperature"], int(seed))
        cache.set_top_k(case["top_k"])
    context, ids, last = _tokens(case, seed)
    if len(context):
        gh.prefill(model, cache, context, want_logits=False)
    return {"case": case, "model": model, "cache": cache, "ids": ids, "last": last}


# ------------------------------------------------------------------ one pass
def run(state):
    case = state["case"]
    if case["kind"] == "matvec":
        gh.check(gh.lib().gh_q4_0_matvec(state["w"].h, ctypes.c_void_p(state["x"].data_ptr()),
                                         ctypes.c_void_p(state["y"].data_ptr()), int(case["softcap"]), 30.0))
        return {"y": state["y"]}
    if case["kind"] == "attention":
        gh.check(gh.lib().gh_attention_decode(_context().h, ctypes.c_void_p(state["q"].data_ptr()),
                                              ctypes.c_void_p(state["k"].data_ptr()),
                                              ctypes.c_void_p(state["v"].data_ptr()), case["heads"],
                                              case["kv_heads"], case["head_dim"], case["begin"], case["end"], 0,
                                              ctypes.c_void_p(state["out"].data_ptr())))
        return {"out": state["out"]}
    model, cache = state["model"], state["cache"]
    cache.truncate(case["start"])  # the next pass continues from the same context
    if case["kind"] == "step":
        logits, _, token = gh.runGemmaInferenceCached(model, int(state["ids"][0]), cache)
        return {"logits": logits, "token": token}
    if case["kind"] == "prefill":
        logits, _, token = gh.prefill(model, cache, state["ids"])
        return {"logits": logits}
    ids = gh.generate(model, cache, state["ids"], case["new"])
    logits, _, _ = gh.runGemmaInferenceCached(model, state["last"], cache)
    return {"ids": ids, "logits": logits}


# ------------------------------------------------------------------ what a pass cannot do without
def _layer_weights(case):
    H, nq, nkv, hd, F = SHAPES[case["model"]][:5]
    return (nq + 2 * nkv) * hd * H + nq * hd * H + 3 * F * H


def _attended(case, first, n):
    """Cache rows met by the queries at positions first .. first+n-1, summed over the layers: (distinct rows, pairs)."""
    window, every = SHAPES[case["model"]][6:8]
    rows = pairs = 0
    for layer in range(case["layers"]):
        full = every == 0 or (layer + 1) % every == 0 or window == 0
        pairs += sum(min(p + 1, p + 1 if full else window) for p in range(first, first + n))
        rows += first + n if full else min(first + n, window + n)
    return rows, pairs


def work(case):
    if case["kind"] == "matvec":
        n = case["rows"] * case["cols"]
        return {"bytes": n / 32 * 18 + 4 * (case["rows"] + case["cols"]), "flops": 2 * n}
    if case["kind"] == "attention":
        n, hd = case["end"] - case["begin"], case["head_dim"]
        return {"bytes": 8 * n * case["kv_heads"] * hd + 8 * case["heads"] * hd, "flops": 4 * n * case["heads"] * hd}
    H, nq, nkv, hd, F, V = SHAPES[case["model"]][:6]
    per = 18 / 32 if case["weights"] == "q4_0" else 4
    body, head = case["layers"] * _layer_weights(case), V * H
    if case["kind"] == "prefill":
        rows, pairs = _attended(case, case["start"], case["tokens"])
        return {"bytes": per * (body + head) + 8 * rows * nkv * hd + 4 * V,
                "flops": 2 * case["tokens"] * body + 2 * head + 4 * pairs * nq * hd}
    # one step per token: every prompt token but the last gives one, then each new one, then the closing step
    steps = 1 if case["kind"] == "step" else case["tokens"] + case["new"]
    pairs = _attended(case, case["start"], steps)[1]
    return {"bytes": steps * per * (body + head) + 8 * pairs * nkv * hd + 4 * V,
            "flops": 2 * steps * (body + head) + 4 * pairs * nq * hd}


def tolerance(case):
    # about four times what two f32 implementations differ by: each measures 0.7e-7 (matvec), 1.9e-7 (attention)
    # and 0.4e-6 to 1.6e-6 (logits, f32 rounding carried through all layers) from the 64-bit result
    if case["kind"] == "matvec":
        return {"rel": 6e-7}
    if case["kind"] == "attention":
        return {"rel": 1e-6}
    return {"rel": 6e-6}


# ------------------------------------------------------------------ the same in 64 bits
def _norm(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * (1.0 + w)


def _rope(x, pos, theta):
    """Split-half rotation of x [n, heads, hd]; the angle is the f32 product of position and f32 frequency, which is
    how the model defines it."""
    half = x.shape[-1] // 2
    power = np.power(np.float64(np.float32(theta)), np.arange(half) * 2.0 / (2 * half)).astype(np.float32)
    freq = np.float32(1.0) / power
    angle = torch.from_numpy(pos.astype(np.float32)[:, None] * freq[None, :]).cuda().double()
    c, s = torch.cos(angle)[:, None, :], torch.sin(angle)[:, None, :]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * s, a * s + b * c], dim=-1)


class _Exact:
    def __init__(self, case, seed):
        self.case, self.t = case, {}
        for name, is_matrix, t in _tensors(case, _generator(seed)):
            self.t[name] = _q4_values(t) if is_matrix and case["weights"] == "q4_0" else t.double()
        self.k, self.v = [None] * case["layers"], [None] * case["layers"]

    def forward(self, ids, pos0):
        """Logits after the last of the tokens `ids` at positions pos0 .. ."""
        H, nq, nkv, hd, F, V, window, every, local, glob, _ = SHAPES[self.case["model"]]
        n, t = len(ids), self.t
        x = t["token_embd.weight"][torch.as_tensor(ids, device="cuda", dtype=torch.long)] * math.sqrt(H)
        pos = np.arange(pos0, pos0 + n)
        at = torch.from_numpy(pos).cuda()[:, None]
        for layer in range(self.case["layers"]):
            w = lambda name: t["blk.%d.%s.weight" % (layer, name)]  # noqa: E731, B023
            full = every == 0 or (layer + 1) % every == 0
            y = _norm(x, w("attn_norm"))
            q = _norm((y @ w("attn_q").t()).view(n, nq, hd), w("attn_q_norm"))
            k = _norm((y @ w("attn_k").t()).view(n, nkv, hd), w("attn_k_norm"))
            v = (y @ w("attn_v").t()).view(n, nkv, hd)
            q, k = _rope(q, pos, glob if full else local), _rope(k, pos, glob if full else local)
            old_k, old_v = self.k[layer], self.v[layer]
            self.k[layer] = k = k if old_k is None else torch.cat([old_k, k])
            self.v[layer] = v = v if old_v is None else torch.cat([old_v, v])
            key = torch.arange(len(k), device="cuda")[None, :]
            hidden = key > at
            if window and not full:
                hidden = hidden | (key <= at - window)
            heads = []
            for h in range(nq):
                g = h // (nq // nkv)
                s = (q[:, h].contiguous() @ k[:, g].t().contiguous()) / math.sqrt(hd)
                heads.append(torch.softmax(s.masked_fill_(hidden, -math.inf), -1) @ v[:, g].contiguous())
            x = x + _norm(torch.cat(heads, -1) @ w("attn_output").t(), w("post_attention_norm"))
            y = _norm(x, w("ffn_norm"))
            a = y @ w("ffn_gate").t()
            z = torch.clamp(0.7978845608 * (a + 0.044715 * a * a * a), -10.0, 10.0)
            y = 0.5 * a * (1.0 + torch.tanh(z)) * (y @ w("ffn_up").t())
            x = x + _norm(y @ w("ffn_down").t(), w("post_ffw_norm"))
        return t["token_embd.weight"] @ _norm(x[-1], t["output_norm.weight"])


def exact(case, seed):
    if case["kind"] == "matvec":
        g = _generator(seed)
        w = _q4_values(_q4_blocks(g, case["rows"], case["cols"]))
        y = w @ torch.randn(case["cols"], generator=g, device="cuda").double()
        return {"y": 30.0 * torch.tanh(y / 30.0) if case["softcap"] else y}
    if case["kind"] == "attention":
        q, k, v = (x.double() for x in _attention_inputs(case, seed))
        nq, nkv, hd = case["heads"], case["kv_heads"], case["head_dim"]
        q, k, v = q.view(nq, hd), k.view(-1, nkv, hd)[case["begin"]:], v.view(-1, nkv, hd)[case["begin"]:]
        out = []
        for h in range(nq):
            g = h // (nq // nkv)
            p = torch.softmax(k[:, g].contiguous() @ q[h] / math.sqrt(hd), 0)
            out.append(p @ v[:, g].contiguous())
        return {"out": torch.cat(out)}
    m = _Exact(case, seed)
    context, ids, last = _tokens(case, seed)
    at = case["start"]
    if len(context):
        m.forward(context, 0)
    logits = m.forward(ids, at)
    if case["kind"] == "step":
        return {"logits": logits, "token": None}
    if case["kind"] == "prefill":
        return {"logits": logits}
    at += len(ids)
    for _ in range(case["new"] - 1):
        logits = m.forward([int(torch.argmax(logits))], at)
        at += 1
    return {"ids": None, "logits": m.forward([last], at)}
