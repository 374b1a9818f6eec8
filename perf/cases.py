"""The token loop's performance cases: what a program that serves Llama-family models has this library do, each through
the public calls of qpack_amd.HipLlama (qp::Model's methods) on a model that it has already loaded.

The models are the benchmark shapes of qpack_amd.synth.CONFIGS: the 0.5B ones whole, the 8B and 7B ones as a slice of
eight layers with the whole output head (the layers repeat; eight of them are far larger than any cache), the head tied
to the embedding so that a state holds one copy of it.  Weights are N(0, 0.02) quantised by the rules of the file format.
"""
import ctypes as C
import math

import numpy as np
import torch

from qpack_amd import HipLlama, _lib, synth

STD = 0.02


def _model(key, layers):
    s = synth.CONFIGS[key]
    return {"hidden": s.hidden, "layers": layers or s.layers, "heads": s.heads, "kv_heads": s.kv_heads,
            "head_dim": s.head_dim, "ffn": s.ffn, "vocab": s.vocab, "bias": s.qkv_bias, "theta": s.rope_theta,
            "eps": s.rms_eps, "q4": s.q4, "q4m": s.q4m_alt, "q1": s.mlp_q1}


MODELS = {
    "05b_q8": _model("c1", 0),
    "05b_q4": _model("c2", 0),
    "8b_q8": _model("c3", 8),
    "7b_q4m": _model("c5", 8),
    "8b_q1": _model("c3_q1", 8),
}


def listed():
    return [
        # a short completion of the small model, picked greedily on the device: launches and latency
        {"name": "greedy_05b_q8", "model": "05b_q8", "op": "greedy", "ctx": 32, "n": 16, "m": 0},
        # one token for a sampler that takes its candidates from the device: the smallest call there is
        {"name": "topk_05b_q4", "model": "05b_q4", "op": "topk", "ctx": 700, "n": 1, "m": 40},
        # the ordinary chat answer of the 8B model after a prompt of about a hundred tokens
        {"name": "greedy_8b_q8", "model": "8b_q8", "op": "greedy", "ctx": 137, "n": 16, "m": 0},
        # token by token with every logits vector on the host (a host sampler), some way into a conversation
        {"name": "step_8b_q8", "model": "8b_q8", "op": "step", "ctx": 1500, "n": 4, "m": 0},
        # decoding behind a long document, 4-bit weights
        {"name": "greedy_7b_q4m_16k", "model": "7b_q4m", "op": "greedy", "ctx": 16384, "n": 16, "m": 0},
        # one line of chat to the small model
        {"name": "prompt_05b_q8", "model": "05b_q8", "op": "prompt", "ctx": 0, "n": 33, "m": 0},
        # a page of prompt to the small 4-bit model, whose state the server keeps for the prompts that start alike
        {"name": "prompt_05b_q4", "model": "05b_q4", "op": "save", "ctx": 0, "n": 512, "m": 0},
        # a short question to the 8B model
        {"name": "prompt_8b_q8_short", "model": "8b_q8", "op": "prompt", "ctx": 0, "n": 77, "m": 0},
        # a long prompt to the 8B model: the largest call
        {"name": "prompt_8b_q8_long", "model": "8b_q8", "op": "prompt", "ctx": 0, "n": 2048, "m": 0},
        # the next turn of a conversation that is already long: few new tokens, many cached ones
        {"name": "turn_7b_q4m", "model": "7b_q4m", "op": "prompt", "ctx": 12000, "n": 150, "m": 0},
        # speculative decoding: one token and seven drafts checked in one call, logits of every position
        {"name": "verify_8b_q8", "model": "8b_q8", "op": "verify", "ctx": 600, "n": 8, "m": 0},
        # a prompt to a model with 1-bit MLP matrices
        {"name": "prompt_8b_q1", "model": "8b_q1", "op": "prompt", "ctx": 0, "n": 300, "m": 0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["greedy", "topk", "step", "prompt", "prompt", "verify", "save"])
    case = {"model": rng.choice(sorted(MODELS)), "op": op, "m": 0}
    if op == "prompt":
        case["n"] = _log_int(rng, 2, 2048)
        case["ctx"] = rng.choice([0, _log_int(rng, 16, 16384)])
    elif op == "save":
        case["n"] = _log_int(rng, 16, 1024)
        case["ctx"] = 0
    elif op == "verify":
        case["n"] = rng.randint(2, 16)
        case["ctx"] = _log_int(rng, 16, 4096)
    else:
        case["n"] = rng.randint(4, 16) if op == "greedy" else rng.randint(1, 8)
        case["ctx"] = _log_int(rng, 16, 16384)
        if op == "topk":
            case["m"] = _log_int(rng, 1, 128)
    limit = max(listed(), key=lambda c: work(c)["flops"])
    while work(case)["flops"] > work(limit)["flops"] or (case["model"] == "8b_q1" and case["n"] > 1024):
        case["n"] = case["n"] * 3 // 4
    return case


# ---------------------------------------------------------------- the model of a case
def _kinds(m, l):
    """the layer's matrices: name, rows, columns, kind (the policies of qpack_amd.synth)"""
    d, ff, qd, kvd = m["hidden"], m["ffn"], m["heads"] * m["head_dim"], m["kv_heads"] * m["head_dim"]
    att = "q4" if m["q4"] else "q8"
    mlp = "q1" if m["q1"] else att
    wide = "q8" if m["q4m"] else att
    down = "q8" if m["q4m"] and l % 2 == 0 else mlp
    return [("wq", qd, d, att), ("wk", kvd, d, att), ("wv", kvd, d, wide), ("wo", d, qd, att), ("w_gate", ff, d, mlp),
            ("w_up", ff, d, mlp), ("w_down", d, ff, down)]


def _quantise(w, kind):
    """(stored bytes, stored scale) of a float matrix in the file's layout"""
    rows, cols = w.shape
    if kind == "q8":
        s = w.abs().amax(1) / 127
        return torch.round(w / s[:, None]).clamp_(-127, 127).to(torch.int8), s
    if kind == "q4":   # byte j of a 32-column group: column j low, column j + 16 high, each stored as q + 8
        g = w.view(rows, cols // 32, 32)
        s = (g.abs().amax(2) / 7).half()
        q = torch.round(g / s.float()[:, :, None]).clamp_(-8, 7).to(torch.int32) + 8
        return (q[:, :, :16] | (q[:, :, 16:] << 4)).to(torch.uint8).view(rows, cols // 2), s
    g = w.view(rows, cols // 128, 128)   # q1: sign bits, least significant first; the group's mean magnitude
    bits = (g >= 0).to(torch.int32).view(rows, cols // 8, 8)
    q = (bits << torch.arange(8, device=w.device, dtype=torch.int32)).sum(2).to(torch.uint8)
    return q, g.abs().mean(2).half()


def _dequantise(q, s, kind):
    rows = q.shape[0]
    if kind == "q8":
        return q.double() * s.double()[:, None]
    if kind == "q4":
        b = q.view(rows, -1, 16).to(torch.int32)
        return ((torch.cat((b & 15, b >> 4), 2) - 8).double() * s.double()[:, :, None]).view(rows, -1)
    bits = (q.to(torch.int32)[:, :, None] >> torch.arange(8, device=q.device, dtype=torch.int32)) & 1
    return ((2 * bits - 1).view(rows, -1, 128).double() * s.double()[:, :, None]).view(rows, -1)


def _tensors(m, gen):
    """every tensor of the model, in order: (name, kind, stored, scale) on the GPU"""
    def normal(*shape):
        return torch.randn(*shape, device="cuda", generator=gen)

    yield ("embed", "q8", *_quantise(normal(m["vocab"], m["hidden"]) * STD, "q8"))
    yield ("final_norm", "f32", 1 + 0.1 * normal(m["hidden"]), None)
    for l in range(m["layers"]):
        p = f"layers.{l}."
        for name in ("attn_norm", "ffn_norm"):
            yield (p + name, "f32", 1 + 0.1 * normal(m["hidden"]), None)
        for name, rows, cols, kind in _kinds(m, l):
            yield (p + name, kind, *_quantise(normal(rows, cols) * STD, kind))
            if m["bias"] and name in ("wq", "wk", "wv"):
                yield (p + "b" + name[1], "f32", normal(rows) * STD, None)


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _cache(m, ctx, seed):
    """fp16 N(0, 1) cache rows of `ctx` positions, [layers][k, v][ctx][kv heads x head dim]"""
    shape = (m["layers"], 2, ctx, m["kv_heads"] * m["head_dim"])
    return torch.randn(*shape, device="cuda", generator=_generator(seed + 1)).half()


def _tokens(case, seed):
    n = 1 if case["op"] == "greedy" else case["n"]
    return np.random.default_rng(seed + 2).integers(0, MODELS[case["model"]]["vocab"], n).astype(np.int32)


def prepare(case, seed):
    m = MODELS[case["model"]]
    kinds = {"f32": _lib.QPH_F32, "q8": _lib.QPH_Q8, "q4": _lib.QPH_Q4, "q1": _lib.QPH_Q1}
    entries, keep = [], []
    for name, kind, q, s in _tensors(m, _generator(seed)):
        q = q.cpu().contiguous()
        s = s.cpu().contiguous() if s is not None else None
        keep.append((q, s))
        rows = q.shape[0]
        cols = 1 if kind == "f32" else q.shape[1] * {"q8": 1, "q4": 2, "q1": 8}[kind]
        entries.append(_lib.Tensor(name.encode(), kinds[kind], rows, cols, q.data_ptr(), s.data_ptr() if s is not None else None, 0, 0))
    cfg = _lib.Config(m["hidden"], m["layers"], m["heads"], m["kv_heads"], m["head_dim"], m["ffn"], m["vocab"], 1,
                      int(m["bias"]), 32768, m["eps"], m["theta"])
    need = case["ctx"] + case["n"] + 1
    handle = C.c_void_p()
    _lib.check(_lib.lib().qph_create(C.byref(cfg), (_lib.Tensor * len(entries))(*entries), len(entries),
                                     4096 if need <= 4096 else 20480, C.byref(handle)))
    model = HipLlama(handle.value)
    if case["ctx"]:
        model.restore(np.int32(case["ctx"]).tobytes() + _cache(m, case["ctx"], seed).cpu().numpy().tobytes())
    torch.cuda.empty_cache()
    return {"case": case, "model": model, "tokens": _tokens(case, seed)}


def run(state):
    case, model, toks = state["case"], state["model"], state["tokens"]
    model.rewind(case["ctx"])
    if case["op"] == "prompt":
        return model.prefill(toks)
    if case["op"] == "save":
        logits = model.prefill(toks)
        return logits, np.frombuffer(model.snapshot(), np.float16, offset=4)
    if case["op"] == "verify":
        return model.prefill_all(toks)
    if case["op"] == "step":
        return [model.step(int(t)) for t in toks]
    if case["op"] == "topk":
        return [model.step_topk(int(t), case["m"]) for t in toks]
    picked = model.greedy_run(int(toks[0]), case["n"])
    return picked, model.step(int(picked[-1]))


def work(case):
    m, n, ctx = MODELS[case["model"]], case["n"], case["ctx"]
    per_weight = {"q8": 1.0, "q4": 0.5 + 2 / 32, "q1": 0.125 + 2 / 128}
    mats = [k for l in range(m["layers"]) for k in _kinds(m, l)]
    layer_bytes = sum(r * c * per_weight[k] for _, r, c, k in mats)
    layer_params = sum(r * c for _, r, c, _ in mats)
    head = m["vocab"] * m["hidden"]
    kvd, qd = m["kv_heads"] * m["head_dim"], m["heads"] * m["head_dim"]
    tokens = n + 1 if case["op"] == "greedy" else n
    # a token of a sequential loop needs every weight and the whole cache again; a batch needs them once
    passes = tokens if case["op"] in ("greedy", "step", "topk") else 1
    heads = 1 if case["op"] in ("prompt", "save") else tokens
    seen = tokens * ctx + tokens * (tokens + 1) / 2   # (token, attended position) pairs
    cached = seen if passes > 1 else ctx + tokens
    out = 8 * case["m"] * n if case["m"] else 4 * m["vocab"] * (1 if case["op"] in ("prompt", "greedy", "save") else n)
    if case["op"] == "save":
        out += 4 * m["layers"] * kvd * tokens
    return {"bytes": passes * (layer_bytes + head) + 4 * m["layers"] * kvd * cached + out,
            "flops": 2.0 * layer_params * tokens + 2.0 * head * heads + 4.0 * m["layers"] * qd * seen}


def tolerance(case):
    # the reference's order of operations against this library's own: 1e-4 to 4e-4 and 2e-4 to 2e-3, most of it cache rows
    # and activations that round to the next 16-bit value and travel on through the layers
    t = {"rel": 1.5e-3, "max": 8e-3}
    if case["op"] == "greedy":
        t["differ"] = 0.1
    if case["op"] == "topk":   # neighbours in the order of the candidates lie closer together the more there are
        t["differ"] = min(0.6, 0.2 + 0.004 * case["m"])
    return t


# ---------------------------------------------------------------- the same results in 64 bits
def _activation(x):
    """what a quantised matrix multiplies: 16-bit integers per 128 columns (part of the format's arithmetic)"""
    b = x.view(x.shape[0], -1, 128)
    mx = b.abs().amax(2, keepdim=True)
    q = torch.round(b * torch.where(mx > 0, 32767 / mx, torch.zeros_like(mx)))
    return (q * (mx / 32767)).view(x.shape)


class _Exact:
    def __init__(self, case, seed):
        self.m = m = MODELS[case["model"]]
        self.w = {}
        for name, kind, q, s in _tensors(m, _generator(seed)):
            self.w[name] = q.double() if kind == "f32" else _dequantise(q, s, kind)
        self.cache = [[t.double() for t in layer] for layer in _cache(m, case["ctx"], seed)]

    def mat(self, x, name):
        return _activation(x) @ self.w[name].t()

    def norm(self, x, name):
        return x / torch.sqrt((x * x).mean(1, keepdim=True) + self.m["eps"]) * self.w[name]

    def rope(self, x, pos):
        hd = self.m["head_dim"]
        inv = self.m["theta"] ** (-torch.arange(0, hd, 2, device="cuda", dtype=torch.float64) / hd)
        a = (pos.double()[:, None] * inv)[:, None, :]
        x = x.view(x.shape[0], -1, hd)
        lo, hi = x[..., :hd // 2], x[..., hd // 2:]
        return torch.cat((lo * a.cos() - hi * a.sin(), hi * a.cos() + lo * a.sin()), 2)

    def feed(self, toks):
        """logits of every token of `toks`, whose rows join the cache"""
        m, hd, rep = self.m, self.m["head_dim"], self.m["heads"] // self.m["kv_heads"]
        x = self.w["embed"][torch.as_tensor(toks, device="cuda", dtype=torch.long)]
        n, p0 = len(toks), self.cache[0][0].shape[0]
        pos = p0 + torch.arange(n, device="cuda")
        mask = torch.arange(p0 + n, device="cuda")[None, :] > pos[:, None]
        for l in range(m["layers"]):
            p = f"layers.{l}."
            h = self.norm(x, p + "attn_norm")
            q, k, v = (self.mat(h, p + "w" + c) + (self.w[p + "b" + c] if m["bias"] else 0) for c in "qkv")
            q, k = self.rope(q, pos), self.rope(k, pos).reshape(n, -1)
            K, V = (torch.cat((old, new.float().half().double())) for old, new in zip(self.cache[l], (k, v)))
            self.cache[l] = [K, V]
            att = torch.empty_like(q)
            for i in range(m["heads"]):
                g = slice((i // rep) * hd, (i // rep + 1) * hd)
                s = (q[:, i] @ K[:, g].t()) / math.sqrt(hd)
                att[:, i] = torch.softmax(s.masked_fill_(mask, -math.inf), 1) @ V[:, g]
            x = x + self.mat(att.reshape(n, -1), p + "wo")
            h = self.norm(x, p + "ffn_norm")
            gate = self.mat(h, p + "w_gate")
            x = x + self.mat(gate * torch.sigmoid(gate) * self.mat(h, p + "w_up"), p + "w_down")
        return x

    def head(self, x):
        return self.mat(self.norm(x, "final_norm"), "embed")


def exact(case, seed):
    e, toks = _Exact(case, seed), _tokens(case, seed)
    host = lambda t: t.cpu().numpy()
    if case["op"] == "prompt":
        return host(e.head(e.feed(toks)[-1:])[0])
    if case["op"] == "save":
        logits = host(e.head(e.feed(toks)[-1:])[0])
        return logits, np.concatenate([host(t).ravel() for layer in e.cache for t in layer])
    if case["op"] == "verify":
        return host(e.head(e.feed(toks)))
    if case["op"] == "step":
        return [host(r) for r in e.head(e.feed(toks))]
    if case["op"] == "topk":
        out = []
        for r in e.head(e.feed(toks)):
            val, idx = torch.sort(r, descending=True, stable=True)
            out.append((host(idx[:case["m"]]).astype(np.int32), host(val[:case["m"]])))
        return out
    picked, tok = [], int(toks[0])
    for _ in range(case["n"]):
        tok = int(e.head(e.feed([tok]))[0].argmax())
        picked.append(tok)
    return np.array(picked, np.int32), host(e.head(e.feed([tok]))[0])
