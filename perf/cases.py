"""The workloads whose speed this library is held to: what a program that serves its models asks of them.

Every case runs through the public Python entry points (``crane_amd.backend.Model`` over the C ABI), on the library's own model
configurations with deterministic synthetic weights.  A program creates a model once and then feeds it inputs: the handle and its cached
context are made by ``prepare``, a pass is what happens per request.

Kinds of pass:

``reply``   one sequence answers behind a cached context, token by token, with the logits of every token, as a program that samples on the
            host reads them.  Dense decoders step one token; decoders with a recurrent state fork the cached context (a shared prefix)
            and step a few.
``prompt``  a whole prompt of one sequence, the logits of its last position.
``round``   decode rounds of a group of sequences with contexts of their own lengths: greedy ids in every round, the logits of the last.
``serve``   mixed steps of a layer-list decoder: many short prompts in one batch, then decode tokens beside portions of one long prompt.
``image``   images through a vision tower.

The greedy ids are an output where rounding cannot tip them: in 8-bit weights a code of the activations, and between bfloat16 rows a
routing choice, moves the logits by more than the two best of random weights are apart, so there the logits alone are compared.

``exact`` restates the decoders and the tower in plain torch float64 on the same weights.
"""
import math

import numpy as np
import torch

from crane_amd import configs
from crane_amd.backend import Model

WEIGHT_SEED = 0
ROUNDS = 4                 # decode rounds of a `round` pass
REPLY = 8                  # tokens of a `reply` pass behind a fork
PORTIONS = 4               # steps over which the long prompt of a `serve` pass is spread
LONGEST = 4608             # cm_opts.max_seq_len of every handle


def listed():
    return [
        # the smallest call: one token of a small model right after a short question
        {"name": "reply-0.6b-short", "kind": "reply", "model": "qwen3-0.6b", "quant": "none", "context": 75},
        # the benchmark's own workload: one token of the 8B model behind 1024 cached ones, with the logits a host sampler wants
        {"name": "reply-8b", "kind": "reply", "model": "qwen3-8b", "quant": "none", "context": 1024},
        # a chat turn's question: a ragged prompt that fills less than one tile row of every product
        {"name": "prompt-8b-short", "kind": "prompt", "model": "qwen3-8b", "quant": "none", "tokens": 117},
        # a document: more rows than one prompt chunk holds
        {"name": "prompt-8b-long", "kind": "prompt", "model": "qwen3-8b", "quant": "none", "tokens": 2500},
        # serving: 32 running sequences with contexts between a few and a thousand tokens
        {"name": "round-8b-32", "kind": "round", "model": "qwen3-8b", "quant": "none", "sequences": 32, "longest": 1000},
        # the same in 8-bit weights, a smaller group
        {"name": "round-8b-q8-20", "kind": "round", "model": "qwen3-8b", "quant": "q8_0", "sequences": 20, "longest": 700},
        # the hybrid decoder at the prompt length of the published figures
        {"name": "prompt-2b-hybrid", "kind": "prompt", "model": "qwen3.5-2b", "quant": "none", "tokens": 4165},
        # a hybrid decoder's reply behind a shared prefix
        {"name": "reply-0.8b-fork", "kind": "reply", "model": "qwen3.5-0.8b", "quant": "none", "context": 1900},
        # a photo and a ragged smaller picture through the tower of the vision-language model
        {"name": "image-2b", "kind": "image", "model": "qwen3-vl-2b", "quant": "none", "height": 42, "width": 64, "extra": 22},
        # layer-list decoders: a prompt through layers of an 8B-class width with routed experts
        {"name": "prompt-experts-8b", "kind": "prompt", "model": "gizezen-8b-4l", "quant": "none", "tokens": 2048},
        # ... a server's mixed batches on a 24-layer model
        {"name": "serve-experts-1b", "kind": "serve", "model": "gizezen-1b", "quant": "none", "sequences": 24, "longest": 130, "long_prompt": 1210},
        # ... and one conversation's reply on it
        {"name": "reply-experts-1b", "kind": "reply", "model": "gizezen-1b", "quant": "none", "context": 1000},
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["reply", "reply", "prompt", "prompt", "prompt", "round", "round", "image", "serve"])
    if kind == "reply":
        model = rng.choice(["qwen3-0.6b", "qwen3-8b", "qwen3.5-0.8b", "gizezen-1b"])
        return {"kind": kind, "model": model, "quant": "none", "context": _spread(rng, 24, 2048)}
    if kind == "prompt":
        model, quant, most = rng.choice([("qwen3-8b", "none", 2400), ("qwen3-8b", "none", 2400), ("qwen3.5-2b", "none", 4000),
                                         ("gizezen-8b-4l", "none", 2048), ("gizezen-1b", "none", 2048)])
        return {"kind": kind, "model": model, "quant": quant, "tokens": _spread(rng, 24, most)}
    if kind == "round":
        return {"kind": kind, "model": "qwen3-8b", "quant": rng.choice(["none", "q8_0"]), "sequences": _spread(rng, 3, 32),
                "longest": _spread(rng, 60, 900)}
    if kind == "image":
        return {"kind": kind, "model": "qwen3-vl-2b", "quant": "none", "height": 2 * rng.randint(6, 21), "width": 2 * rng.randint(6, 31),
                "extra": 2 * rng.randint(3, 11)}
    return {"kind": kind, "model": "gizezen-1b", "quant": "none", "sequences": rng.randint(3, 24), "longest": _spread(rng, 24, 130),
            "long_prompt": _spread(rng, 64, 1200)}


# ---- inputs ----------------------------------------------------------------------------------------------------------------
def _vocab(cfg):
    return cfg.get("vocab") or cfg.get("vocab_size") or cfg["text_config"]["vocab_size"]


def _layered(cfg):
    return "architecture" in cfg


def _recurrent(cfg):
    return _layered(cfg) or cfg.get("model_type", "").startswith("qwen3_5")


def _inputs(case, seed):
    """Token ids (or pictures) of a case, from the seed alone."""
    rs = np.random.RandomState(seed % (2 ** 32))
    cfg = configs.get_config(case["model"])
    ids = lambda n: rs.randint(0, _vocab(cfg), n).astype(np.uint32)  # noqa: E731
    kind = case["kind"]
    if kind == "reply":
        return {"context": ids(case["context"]), "tokens": ids(REPLY if _recurrent(cfg) else 1)}
    if kind == "prompt":
        return {"prompt": ids(case["tokens"])}
    if kind == "round":
        n, top = case["sequences"], case["longest"]
        lens = [top] + [int(rs.randint(min(16, top), top + 1)) for _ in range(n - 1)]
        return {"contexts": [ids(k) for k in lens], "tokens": [ids(n) for _ in range(ROUNDS)]}
    if kind == "serve":
        n, top = case["sequences"], case["longest"]
        return {"prompts": [ids(int(rs.randint(min(12, top), top + 1))) for _ in range(n)], "long": ids(case["long_prompt"]),
                "tokens": [ids(n) for _ in range(PORTIONS)]}
    grid = [(1, case["height"], case["width"]), (1, case["extra"], case["extra"])]
    rows = sum(t * h * w for t, h, w in grid)
    v = cfg["vision_config"]
    px = rs.standard_normal((rows, v["in_channels"] * v["temporal_patch_size"] * v["patch_size"] ** 2))
    return {"grid": grid, "pixels": np.clip(0.6 * px, -1, 1).astype(np.float32)}


_HELD = {}                 # the model a program is serving: one handle, created once


def _model(case):
    key = (case["model"], case["quant"])
    if key not in _HELD:
        _HELD.clear()
        cfg = configs.get_config(case["model"])
        kw = dict(max_seq_len=LONGEST, max_seqs=160, kv_pool_tokens=160 * 1024, isq=None if case["quant"] == "none" else case["quant"])
        _HELD[key] = Model.synthetic(cfg, seed=WEIGHT_SEED, **kw)
    return _HELD[key]


class _State:
    """A request's sequences on the handle, given back with it."""

    def __init__(self, case, model, given):
        self.case, self.model, self.given, self.seqs = case, model, given, []

    def sequence(self):
        s = self.model.seq_alloc()
        self.seqs.append(s)
        return s

    def __del__(self):
        for s in self.seqs:
            try:
                self.model.seq_free(s)
            except Exception:
                pass


def prepare(case, seed):
    given, model = _inputs(case, seed), _model(case)
    st = _State(case, model, given)
    kind = case["kind"]
    if kind == "reply":
        model.seq_forward(st.sequence(), given["context"], 0, want_logits=False)
    elif kind == "prompt":
        st.sequence()
    elif kind == "round":
        pending = [(st.sequence(), c) for c in given["contexts"]]
        while pending:                                     # as many whole prompts as one pass takes
            take, rows = [], 0
            while pending and rows + len(pending[0][1]) <= 2048:
                rows += len(pending[0][1])
                take.append(pending.pop(0))
            model.prefill_batch([s for s, _ in take], [c for _, c in take], want_logits=False)
    elif kind == "serve":
        for _ in range(case["sequences"] + 1):
            st.sequence()
    return st


def _steady(case):
    return case["quant"] == "none" and not _layered(configs.get_config(case["model"]))


def run(state):
    out = _pass(state)
    if not _steady(state.case):
        out.pop("ids", None)
    return out


def _pass(state):
    case, m, given, seqs = state.case, state.model, state.given, state.seqs
    kind = case["kind"]
    if kind == "reply":
        at = len(given["context"])
        if len(given["tokens"]) == 1:
            logits, top = m.seq_forward(seqs[0], given["tokens"], at)
            return {"logits": logits, "ids": [top]}
        f, got, logits = m.seq_fork(seqs[0]), [], []
        for i in range(len(given["tokens"])):
            row, top = m.seq_forward(f, given["tokens"][i:i + 1], at + i)
            logits.append(row)
            got.append(top)
        m.seq_free(f)
        return {"logits": logits, "ids": got}
    if kind == "prompt":
        logits, top = m.seq_forward(seqs[0], given["prompt"], 0)
        return {"logits": logits, "ids": [top]}
    if kind == "round":
        got, logits = [], None
        for i, toks in enumerate(given["tokens"]):
            logits, ids = m.step_batch_decode(seqs, toks, want_logits=i == len(given["tokens"]) - 1)
            got.append(ids)
        for s, c in zip(seqs, given["contexts"]):
            m.seq_truncate(s, len(c))
        return {"logits": logits, "ids": got}
    if kind == "serve":
        for s in seqs:
            m.seq_truncate(s, 0)
        n, long, got, logits = len(seqs) - 1, given["long"], [], None
        _, ids = m.step_batch([(s, p, None) for s, p in zip(seqs, given["prompts"])], want_logits=False)
        got.append(ids)
        cuts = [len(long) * i // PORTIONS for i in range(PORTIONS + 1)]
        for i, toks in enumerate(given["tokens"]):
            items = [(s, toks[k:k + 1], None) for k, s in enumerate(seqs[:n])]
            items.append((seqs[n], long[cuts[i]:cuts[i + 1]], None if i == PORTIONS - 1 else []))
            logits, ids = m.step_batch(items, want_logits=i == PORTIONS - 1)
            got.append(ids)
        return {"logits": logits, "ids": got}
    return {"features": m.encode_images(given["pixels"], given["grid"])}


# ---- what a pass cannot do without -----------------------------------------------------------------------------------------
def _sizes(case):
    """(bytes of a weight, elements read whatever the rows, flops per row, cached elements per token, attention layers, q width, window)."""
    cfg = configs.get_config(case["model"])
    wb = 2.0 if case["quant"] == "none" else 34.0 / 32.0
    if _layered(cfg):
        W, read, per_row, kv, layers = cfg["width"], 0, 0, 0, 0
        for ly in cfg["layers"]:
            mx, ml = ly["mixer"], ly["mlp"]
            own = 0 if "kv_from" in mx else mx["kv_heads"] * (mx["dim"] + mx["vdim"])
            w = W * (mx["heads"] * (mx["dim"] + mx["vdim"] + 1) + own)
            sh = 3 * W * ml["shared"]["ff"] if "shared" in ml else 0
            read += w + sh + 3 * W * ml["expert"]["ff"] * ml["router"]["experts"] + W * (ml["router"]["experts"] + 1)
            per_row += 2 * (w + sh + 3 * W * ml["expert"]["ff"] * ml["router"]["top"] + W * (ml["router"]["experts"] + 1))
            kv, layers = kv + own, layers + 1
        mx = cfg["layers"][0]["mixer"]
        return wb, read, per_row, kv, layers, mx["heads"] * mx["dim"], mx["mask"]["size"], 3 * W * cfg["layers"][0]["mlp"]["expert"]["ff"]
    H, I, L = cfg["hidden_size"], cfg["intermediate_size"], cfg["num_hidden_layers"]
    Hq, Hkv, D = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"]
    if _recurrent(cfg):
        full = L // cfg["full_attention_interval"]
        kd, vd = cfg["linear_num_key_heads"] * cfg["linear_key_head_dim"], cfg["linear_num_value_heads"] * cfg["linear_value_head_dim"]
        n = full * (H * D * (3 * Hq + 2 * Hkv)) + (L - full) * H * (2 * kd + 3 * vd) + L * 3 * H * I
        state = (L - full) * 6 * vd * cfg["linear_key_head_dim"]
        return wb, n, 2 * n + state, full * 2 * Hkv * D, full, Hq * D, 1 << 30, 0
    n = L * (H * D * (2 * Hq + 2 * Hkv) + 3 * H * I)
    return wb, n, 2 * n, L * 2 * Hkv * D, L, Hq * D, 1 << 30, 0


def work(case):
    cfg = configs.get_config(case["model"])
    if case["kind"] == "image":
        v = cfg["vision_config"]
        VH, VI, M, O = v["hidden_size"], v["intermediate_size"], v["spatial_merge_size"] ** 2, v["out_hidden_size"]
        P = v["in_channels"] * v["temporal_patch_size"] * v["patch_size"] ** 2
        frames = [case["height"] * case["width"], case["extra"] ** 2]
        N, mergers = sum(frames), 1 + len(v.get("deepstack_visual_indexes", []))
        body, merge = v["depth"] * (4 * VH * VH + 2 * VH * VI) + P * VH, mergers * (VH * M * VH * M + VH * M * O)
        return {"bytes": 2.0 * (body + merge) + 4.0 * N * P + 4.0 * (N // M) * O,
                "flops": 2.0 * N * body + 2.0 * (N // M) * merge + 4.0 * v["depth"] * VH * sum(f * f for f in frames)}
    wb, n, per_row, kv, layers, qw, window, expert = _sizes(case)
    V, W = _vocab(cfg), cfg.get("hidden_size") or cfg["width"]
    steps = {"reply": REPLY if _recurrent(cfg) else 1, "prompt": 1, "round": ROUNDS, "serve": PORTIONS + 1}[case["kind"]]
    g = _inputs(case, 0)
    # (rows of new tokens, first position) of every sequence
    spans = {"reply": lambda: [(steps, len(g["context"]))], "prompt": lambda: [(len(g["prompt"]), 0)],
             "round": lambda: [(ROUNDS, len(c)) for c in g["contexts"]],
             "serve": lambda: [(len(p) + PORTIONS, 0) for p in g["prompts"]] + [(len(g["long"]), 0)]}[case["kind"]]()
    rows = sum(r for r, _ in spans)
    seen = sum(sum(min(window, a + i + 1) for i in range(r)) for r, a in spans)
    heads = {"reply": steps, "prompt": 1, "round": ROUNDS * len(spans), "serve": len(g.get("prompts", [])) * (PORTIONS + 1) + 1}[case["kind"]]
    # a prompt pass reads its keys once, a decode step the whole window of every sequence
    read = seen if case["kind"] in ("reply", "round") else rows
    least = n
    if expert and case["kind"] == "reply":                 # a token reads the matrices of its own experts only
        ml = cfg["layers"][0]["mlp"]["router"]
        least = n - layers * expert * (ml["experts"] - ml["top"])
    out = {"reply": steps, "prompt": 1, "round": len(spans), "serve": len(spans)}[case["kind"]]
    return {"bytes": steps * (wb * least + (2.0 if wb == 2.0 else wb) * V * W) + 2.0 * kv * (read + rows) + 4.0 * out * V,
            "flops": float(rows) * per_row + 2.0 * heads * V * W + 4.0 * qw * seen * layers}


def tolerance(case):
    if case["quant"] != "none":
        # 8-bit codes of the activations: other sums tip codes over, and 36 layers of them move the logits by 0.024 (measured with another split
        # of the sums, and with the products on the vector units)
        return {"rel": 0.03, "max": 0.3}
    if case["model"].startswith("gizezen"):
        return {"rel": 0.008, "max": 0.1}                   # bf16 rows between the products: 0.0017 against exact
    if case["kind"] == "image":
        return {"rel": 3e-5, "max": 5e-4}                   # products of two-part operands: 5e-6 against exact
    if _recurrent(configs.get_config(case["model"])):
        return {"rel": 1e-4, "max": 1e-3, "differ": 0.01}   # most layers cache in 32 bits: 1.5e-5 against exact
    return {"rel": 1e-3, "max": 0.01, "differ": 0.01}       # a 16-bit cache: 2.3e-4 to 3.8e-4 against exact


# ---- the same in 64 bits ---------------------------------------------------------------------------------------------------
_DEV = "cuda"


def _fmix(h):
    h = h ^ (h >> 16)
    h = (h * 0x85EBCA6B) & 0xFFFFFFFF
    h = h ^ (h >> 13)
    h = (h * 0xC2B2AE35) & 0xFFFFFFFF
    return h ^ (h >> 16)


def _weights(name, shape, std, offset=0.0, rows=None):
    """The synthetic checkpoint's tensor `name` (its rows `rows` alone): four hash bytes summed, scaled, rounded to bfloat16."""
    fnv = 0x811C9DC5
    for b in name.encode():
        fnv = ((fnv ^ b) * 0x01000193) & 0xFFFFFFFF
    ts = int(_fmix(fnv ^ ((WEIGHT_SEED * 0x85EBCA6B + 0x1234567) & 0xFFFFFFFF)))
    inner = int(np.prod(shape[1:])) if len(shape) > 1 else 1
    mul = float(np.float32(std / math.sqrt(21845.0)))
    out = []
    index = torch.arange(shape[0], device=_DEV) if rows is None else rows
    for part in index.split(max(1, (1 << 26) // inner)):
        i = (part[:, None] * inner + torch.arange(inner, device=_DEV)[None, :]) & 0xFFFFFFFF
        h = _fmix((i * 0x9E3779B1 + ts) & 0xFFFFFFFF)
        c = (h & 255) + ((h >> 8) & 255) + ((h >> 16) & 255) + (h >> 24) - 510
        out.append((offset + c.float() * mul).bfloat16())
    return torch.cat(out).reshape((index.numel(),) + tuple(shape[1:]))


def _q8(w):
    """bfloat16 rows as blocks of 32 eight-bit codes with a binary16 scale, and back."""
    b = w.float().reshape(w.shape[0], -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127.0
    inv = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    t = b * inv
    q = torch.sign(t) * torch.floor(t.abs() + 0.5)
    return (q.double() * d.half().double()).reshape(w.shape)


def _lin(case, x, name, rows, cols, std=None):
    w = _weights(name, (rows, cols), std or 1.0 / math.sqrt(cols))
    w = _q8(w) if case["quant"] != "none" else w
    out = torch.empty(x.shape[0], rows, dtype=torch.float64, device=_DEV)
    for a in range(0, rows, 1 << 15):                       # a slice of a large head at a time
        out[:, a:a + (1 << 15)] = x @ w[a:a + (1 << 15)].double().T
    return out


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _turn_halves(x, ang):
    """x [T, heads, d]: element i of the first angles turns with element i + half."""
    h = ang.shape[-1]
    c, s = torch.cos(ang.double())[:, None], torch.sin(ang.double())[:, None]
    u, v = x[..., :h], x[..., h:2 * h]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., 2 * h:]], -1)


def _attend(q, k, v, scale, window=1 << 30, plus_one=False, causal=True):
    """q [T, H, d], k, v [T, G, .]: softmax over the last `window` positions (`plus_one`: one joins the denominator)."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    out = torch.empty(T, H, v.shape[-1], dtype=torch.float64, device=_DEV)
    i = torch.arange(T, device=_DEV)
    hide = (i[None, :] > i[:, None]) | (i[:, None] - i[None, :] >= window) if causal else None
    for h in range(H):
        z = q[:, h] @ k[:, h // (H // G)].T * scale
        z = z.masked_fill(hide, -math.inf) if causal else z
        m = z.amax(-1, keepdim=True)
        m = m.clamp(min=0.0) if plus_one else m
        p = torch.exp(z - m)
        den = p.sum(-1, keepdim=True) + (torch.exp(-m) if plus_one else 0.0)
        out[:, h] = (p / den) @ v[:, h // (H // G)]
    return out


def _pieces(spans, f, *xs):
    """f over every sequence's own rows."""
    got, a = [], 0
    for n in spans:
        got.append(f(*[x[a:a + n] for x in xs]))
        a += n
    return torch.cat(got)


def _positions(spans):
    return torch.cat([torch.arange(n, device=_DEV) for n in spans])


def _dense(case, cfg, ids, spans):
    """Residual rows of the dense decoder behind its last norm."""
    H, I = cfg["hidden_size"], cfg["intermediate_size"]
    Hq, Hkv, D, eps = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"], cfg["rms_norm_eps"]
    inv = torch.tensor([1.0 / cfg["rope_theta"] ** (i / D) for i in range(0, D, 2)], dtype=torch.float64, device=_DEV).float()
    ang = _positions(spans).float()[:, None] * inv[None]
    norm = lambda x, name: _rms(x, eps) * _weights(name, (x.shape[-1],), 0.1, 1.0).double()  # noqa: E731
    x = _weights("model.embed_tokens.weight", (cfg["vocab_size"], H), 1.0, rows=ids).double()
    for li in range(cfg["num_hidden_layers"]):
        p = "model.layers.%d." % li
        h = norm(x, p + "input_layernorm.weight")
        q, k, v = (_lin(case, h, p + "self_attn.%s_proj.weight" % n, r * D, H).reshape(-1, r, D) for n, r in (("q", Hq), ("k", Hkv), ("v", Hkv)))
        q = _turn_halves(norm(q, p + "self_attn.q_norm.weight"), ang)
        k = _turn_halves(norm(k, p + "self_attn.k_norm.weight"), ang)
        a = _pieces(spans, lambda q, k, v: _attend(q, k, v, D ** -0.5), q, k, v)
        x = x + _lin(case, a.reshape(-1, Hq * D), p + "self_attn.o_proj.weight", H, Hq * D)
        h = norm(x, p + "post_attention_layernorm.weight")
        g = _silu(_lin(case, h, p + "mlp.gate_proj.weight", I, H)) * _lin(case, h, p + "mlp.up_proj.weight", I, H)
        x = x + _lin(case, g, p + "mlp.down_proj.weight", H, I)
    return norm(x, "model.norm.weight")


def _delta(q, k, v, g, beta):
    """The gated delta rule, token by token: q, k, v [T, heads, .], g (log decay) and beta [T, heads]."""
    state = torch.zeros(q.shape[1], k.shape[2], v.shape[2], dtype=torch.float64, device=_DEV)
    out = torch.empty_like(v)
    dec = torch.exp(g)[:, :, None, None]
    for t in range(q.shape[0]):
        state *= dec[t]
        new = (v[t] - torch.bmm(k[t, :, None], state)[:, 0]) * beta[t, :, None]
        state.baddbmm_(k[t, :, :, None].contiguous(), new[:, None].contiguous())
        out[t] = torch.bmm(q[t, :, None], state)[:, 0]
    return out


def _hybrid(case, cfg, ids):
    """Residual rows of the hybrid decoder (one sequence) behind its last norm."""
    H, I, T = cfg["hidden_size"], cfg["intermediate_size"], ids.numel()
    Hq, Hkv, D, eps = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"], cfg["rms_norm_eps"]
    NK, NV, K, Vd, taps = (cfg["linear_num_key_heads"], cfg["linear_num_value_heads"], cfg["linear_key_head_dim"],
                           cfg["linear_value_head_dim"], cfg["linear_conv_kernel_dim"])
    rope = cfg["rope_parameters"]
    rot, base = int(D * rope["partial_rotary_factor"]), np.float32(rope["rope_theta"])
    inv = np.array([np.float32(1) / np.power(base, np.float32(2 * i) / np.float32(rot), dtype=np.float32) for i in range(rot // 2)], np.float32)
    ang = torch.arange(T, device=_DEV).float()[:, None] * torch.from_numpy(inv).to(_DEV)[None]
    plain = dict(case, quant="none")
    norm = lambda x, name: _rms(x, eps) * (1.0 + _weights(name, (x.shape[-1],), 0.1).double())  # noqa: E731
    x = _weights("model.embed_tokens.weight", (cfg["vocab_size"], H), 1.0, rows=ids).double()
    for li in range(cfg["num_hidden_layers"]):
        p = "model.layers.%d." % li
        h = norm(x, p + "input_layernorm.weight")
        if (li + 1) % cfg["full_attention_interval"] == 0:
            a = p + "self_attn."
            qg = _lin(case, h, a + "q_proj.weight", Hq * D * 2, H).reshape(T, Hq, 2 * D)
            k = _lin(case, h, a + "k_proj.weight", Hkv * D, H).reshape(T, Hkv, D)
            v = _lin(case, h, a + "v_proj.weight", Hkv * D, H).reshape(T, Hkv, D)
            q = _turn_halves(norm(qg[..., :D], a + "q_norm.weight"), ang)
            k = _turn_halves(norm(k, a + "k_norm.weight"), ang)
            y = (_attend(q, k, v, D ** -0.5) * torch.sigmoid(qg[..., D:])).reshape(T, Hq * D)
            x = x + _lin(case, y, a + "o_proj.weight", H, Hq * D)
        else:
            a, C = p + "linear_attn.", 2 * NK * K + NV * Vd
            mixed = _lin(case, h, a + "in_proj_qkv.weight", C, H)
            z = _lin(case, h, a + "in_proj_z.weight", NV * Vd, H).reshape(T, NV, Vd)
            b, d = _lin(plain, h, a + "in_proj_b.weight", NV, H), _lin(plain, h, a + "in_proj_a.weight", NV, H)
            cw = _weights(a + "conv1d.weight", (C, 1, taps), 0.5).double().reshape(C, taps)
            pad = torch.cat([torch.zeros(taps - 1, C, dtype=torch.float64, device=_DEV), mixed])
            mixed = _silu(sum(pad[j:j + T] * cw[:, j] for j in range(taps)))
            unit = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
            q = unit(mixed[:, :NK * K].reshape(T, NK, K)).repeat_interleave(NV // NK, 1) * K ** -0.5
            k = unit(mixed[:, NK * K:2 * NK * K].reshape(T, NK, K)).repeat_interleave(NV // NK, 1)
            v = mixed[:, 2 * NK * K:].reshape(T, NV, Vd)
            g = -torch.exp(_weights(a + "A_log", (NV,), 0.1, -2.0).double()) * torch.log1p(torch.exp(d + _weights(a + "dt_bias", (NV,), 0.1).double()))
            y = _delta(q, k, v, g, torch.sigmoid(b))
            y = _rms(y, eps) * _weights(a + "norm.weight", (Vd,), 0.1, 1.0).double() * _silu(z)
            x = x + _lin(case, y.reshape(T, NV * Vd), a + "out_proj.weight", H, NV * Vd)
        h = norm(x, p + "post_attention_layernorm.weight")
        g = _silu(_lin(case, h, p + "mlp.gate_proj.weight", I, H)) * _lin(case, h, p + "mlp.up_proj.weight", I, H)
        x = x + _lin(case, g, p + "mlp.down_proj.weight", H, I)
    return norm(x, "model.norm.weight")


_STEPS = []                # tables of the layer-list generator's map, applied 1, 2, 4, ... times


def _apply(tables, h):
    return _xor([tables[b][(h >> (8 * b)) & 255] for b in range(8)])


def _xor(parts):
    out = parts[0]
    for p in parts[1:]:
        out = out ^ p
    return out


def _doubling(level):
    """Byte tables of 2^level steps of the shift-register generator (a linear map over bits)."""
    if not _STEPS:
        bits = (torch.ones(64, dtype=torch.int64) << torch.arange(64)).to(_DEV)
        h = bits ^ (bits << 13)
        h = h ^ ((h >> 7) & ((1 << 57) - 1))
        _STEPS.append(_tables(h ^ (h << 17)))
    while len(_STEPS) <= level:
        t = _STEPS[-1]
        bits = (torch.ones(64, dtype=torch.int64) << torch.arange(64)).to(_DEV)
        _STEPS.append(_tables(_apply(t, _apply(t, bits))))
    return _STEPS[level]


def _tables(image):
    """image[i]: where bit i goes -> eight tables of 256 words."""
    made = []
    for b in range(8):
        t = torch.zeros(256, dtype=torch.int64, device=_DEV)
        for i in range(8):
            t = torch.where((torch.arange(256, device=_DEV) >> i) & 1 == 1, t ^ image[8 * b + i], t)
        made.append(t)
    return made


def _streams(names, n, scale, offset=0.0):
    """The layer-list decoders' synthetic tensors `names` of n elements each, as float32 [names, n]."""
    start = []
    for name in names:
        h = 1469598103934665603 ^ WEIGHT_SEED
        for b in name.encode():
            h = ((h ^ b) * 1099511628211) & 0xFFFFFFFFFFFFFFFF
        start.append(h - (1 << 64) if h >> 63 else h)
    h, level = _apply(_doubling(0), torch.tensor(start, dtype=torch.int64, device=_DEV)[:, None]), 0
    while h.shape[1] < n:
        more = h[:, :n - h.shape[1]]
        t = _doubling(level)
        h = torch.cat([h, torch.cat([_apply(t, x) for x in more.split(1 << 22, 1)], 1)], 1)
        level += 1
    out = torch.empty(h.shape, dtype=torch.float32, device=_DEV)
    for a in range(0, n, 1 << 24):
        x = h[:, a:a + (1 << 24)]
        c = (x & 255) + ((x >> 8) & 255) + ((x >> 16) & 255) + ((x >> 24) & 255) - 510
        out[:, a:a + (1 << 24)] = offset + (c.float() * float(np.float32(scale))) / float(np.float32(147.8))
    return out


def _experts_decoder(cfg, ids, spans):
    """Residual rows of the layer-list decoder with tanh norms and routed experts behind its last norm."""
    W, eps = cfg["width"], cfg["norm"]["eps"]
    ws, n, pos = W ** -0.5, ids.numel(), _positions(spans)
    mat = lambda name, r, c, s=None: _streams([name], r * c, s or c ** -0.5)[0].bfloat16().double().reshape(r, c)  # noqa: E731

    def norm(x, name):
        w, b, a = _streams([name], W, 0.1, 1.0)[0], _streams([name + ".b"], W, 0.1)[0], _streams([name + ".alpha"], 1, 0.05, 0.5)[0]
        return torch.tanh(a.double() * x) * w.double() + b.double()

    def conv(x, name, taps):
        w = _streams([name + ".conv"], x.shape[1] * taps, taps ** -0.5)[0].double().reshape(-1, taps)
        one = lambda p: sum(torch.cat([torch.zeros(taps - 1, p.shape[1], dtype=torch.float64, device=_DEV), p])[j:j + p.shape[0]] * w[:, j]  # noqa: E731
                            for j in range(taps))
        return _pieces(spans, one, x)

    def angles(rot):
        f, sc = [rot["base"] ** (-2.0 * i / rot["dims"]) for i in range(rot["dims"] // 2)], rot.get("scaling")
        for i, fi in enumerate(f if sc else []):
            wave = 2 * math.pi / fi
            if wave > sc["original"] / sc["low"]:
                f[i] = fi / sc["factor"]
            elif wave >= sc["original"] / sc["high"]:
                t = (sc["original"] / wave - sc["low"]) / (sc["high"] - sc["low"])
                f[i] = (1 - t) * fi / sc["factor"] + t * fi
        return pos.double()[:, None] * torch.tensor(f, dtype=torch.float32, device=_DEV).double()[None]

    def turn(x, ang):
        c, s, y = torch.cos(ang)[:, None], torch.sin(ang)[:, None], x.clone()
        d = 2 * ang.shape[1]
        u, v = x[..., 0:d:2], x[..., 1:d:2]
        y[..., 0:d:2], y[..., 1:d:2] = u * c - v * s, v * c + u * s
        return y

    emb = _streams(["embed"], cfg["vocab"] * W, 1.0)[0].reshape(-1, W)[ids].bfloat16().double()
    x, kept = emb * cfg["embedding"]["scale"], []
    for li, ly in enumerate(cfg["layers"]):
        p, mx, ml = "l%d." % li, ly["mixer"], ly["mlp"]
        Hh, G, d, e, taps = mx["heads"], mx["kv_heads"], mx["dim"], mx["vdim"], mx["conv"]
        h, q, ang = norm(x, p + "norm1"), p + "mix.", angles(mx["rot"])
        qs = _rms(turn(conv(h @ mat(q + "q", Hh * d, W).T, q + "q", taps).reshape(n, Hh, d), ang), eps)
        if "kv_from" in mx:
            kv = kept[mx["kv_from"]]
        else:
            kv = (_rms(turn(conv(h @ mat(q + "k", G * d, W).T, q + "k", taps).reshape(n, G, d), ang), eps),
                  conv(h @ mat(q + "v", G * e, W).T, q + "v", taps).reshape(n, G, e))
        kept.append(kv)
        a = _pieces(spans, lambda u, k, v: _attend(u, k, v, mx["scale"], mx["mask"]["size"], True), qs, *kv)
        a = (a * torch.sigmoid(h @ mat(q + "g", Hh, W).T)[:, :, None]).reshape(n, Hh * e)
        x = x + cfg["residual_mult"] * (a @ mat(q + "o", W, Hh * e).T)
        h, ff, E, top = norm(x, p + "norm2"), ml["expert"]["ff"], ml["router"]["experts"], ml["router"]["top"]
        zc, sel = torch.topk(h @ mat(p + "mlp.router", E, W).T, top, -1)
        w, out = torch.softmax(zc, -1), torch.zeros_like(x)
        for j in range(E):
            at, slot = torch.nonzero(sel == j, as_tuple=True)
            if not at.numel():
                continue
            r = "%smlp.e%d." % (p, j)
            gate, up = _streams([r + "gate", r + "up"], ff * W, ws).bfloat16().double().reshape(2, ff, W)
            y = (_silu(h[at] @ gate.T) * (h[at] @ up.T)) @ mat(r + "down", W, ff).T
            out.index_add_(0, at, y * w[at, slot][:, None])
        if "shared" in ml:
            r, sf = p + "mlp.shared.", ml["shared"]["ff"]
            y = (_silu(h @ mat(r + "gate", sf, W).T) * (h @ mat(r + "up", sf, W).T)) @ mat(r + "down", W, sf).T
            out += torch.sigmoid(h @ mat(r + "sg", 1, W).T) * y
        x = x + cfg["residual_mult"] * out
    return norm(x, "final.norm")


def _tower(cfg, pixels, grid):
    """Merged image rows of the vision tower."""
    v = cfg["vision_config"]
    VH, VI, heads, side = v["hidden_size"], v["intermediate_size"], v["num_heads"], int(round(math.sqrt(v["num_position_embeddings"])))
    m, P, hd, p = v["spatial_merge_size"], pixels.shape[1], v["hidden_size"] // v["num_heads"], "model.visual."
    plain = {"quant": "none"}
    lin = lambda x, name, r: _lin(plain, x, name + ".weight", r, x.shape[1]) + _weights(name + ".bias", (r,), 0.1).double()  # noqa: E731

    def ln(x, name):
        y = x - x.mean(-1, keepdim=True)
        return y / torch.sqrt((y * y).mean(-1, keepdim=True) + 1e-6) * _weights(name + ".weight", (x.shape[1],), 0.1, 1.0).double() \
            + _weights(name + ".bias", (x.shape[1],), 0.1).double()

    gelu = lambda x: 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))  # noqa: E731
    table = _weights(p + "pos_embed.weight", (v["num_position_embeddings"], VH), 0.5).double()
    inv = torch.tensor([1.0 / 10000.0 ** (i / (hd // 2)) for i in range(0, hd // 2, 2)], dtype=torch.float64, device=_DEV).float()
    place, ang = [], []
    for _, h, w in grid:                                   # rows of an image in merge-block-major order
        r = torch.arange(h, device=_DEV)[:, None].expand(h, w).reshape(h // m, m, w // m, m).permute(0, 2, 1, 3).reshape(-1)
        c = torch.arange(w, device=_DEV)[None, :].expand(h, w).reshape(h // m, m, w // m, m).permute(0, 2, 1, 3).reshape(-1)
        y = (r.float() * torch.tensor((side - 1) / max(h - 1, 1), device=_DEV)).double()
        z = (c.float() * torch.tensor((side - 1) / max(w - 1, 1), device=_DEV)).double()
        y0, z0 = y.floor().long(), z.floor().long()
        y1, z1 = y.ceil().long().clamp(max=side - 1), z.ceil().long().clamp(max=side - 1)
        dy, dz = (y - y0)[:, None], (z - z0)[:, None]
        place.append(table[y0 * side + z0] * (1 - dy) * (1 - dz) + table[y0 * side + z1] * (1 - dy) * dz
                     + table[y1 * side + z0] * dy * (1 - dz) + table[y1 * side + z1] * dy * dz)
        ang.append(torch.cat([r.float()[:, None] * inv, c.float()[:, None] * inv], -1))
    pw = _weights(p + "patch_embed.proj.weight", (VH, P), P ** -0.5).double()
    x = torch.from_numpy(pixels).to(_DEV).double() @ pw.T + _weights(p + "patch_embed.proj.bias", (VH,), 0.1).double() + torch.cat(place)
    spans, ang = [t * h * w for t, h, w in grid], torch.cat(ang)
    for li in range(v["depth"]):
        b = "%sblocks.%d." % (p, li)
        q, k, u = lin(ln(x, b + "norm1"), b + "attn.qkv", 3 * VH).reshape(-1, 3, heads, hd).unbind(1)
        a = _pieces(spans, lambda q, k, u: _attend(q, k, u, hd ** -0.5, causal=False), _turn_halves(q, ang), _turn_halves(k, ang), u)
        x = x + lin(a.reshape(-1, VH), b + "attn.proj", VH)
        x = x + lin(gelu(lin(ln(x, b + "norm2"), b + "mlp.linear_fc1", VI)), b + "mlp.linear_fc2", VH)
    y = ln(x, p + "merger.norm").reshape(-1, VH * m * m)
    return lin(gelu(lin(y, p + "merger.linear_fc1", VH * m * m)), p + "merger.linear_fc2", v["out_hidden_size"])


@torch.no_grad()
def exact(case, seed):
    global _DEV
    _DEV = "cuda" if torch.cuda.is_available() else "cpu"
    cfg, g, kind = configs.get_config(case["model"]), _inputs(case, seed), case["kind"]
    if kind == "image":
        return {"features": _tower(cfg, g["pixels"], g["grid"])}
    steps = lambda k: [t[k:k + 1] for t in g["tokens"]]  # noqa: E731
    rows = {"reply": lambda: [np.concatenate([g["context"], g["tokens"]])], "prompt": lambda: [g["prompt"]],
            "round": lambda: [np.concatenate([c] + steps(k)) for k, c in enumerate(g["contexts"])],
            "serve": lambda: [np.concatenate([c] + steps(k)) for k, c in enumerate(g["prompts"])] + [g["long"]]}[kind]()
    spans = [len(r) for r in rows]
    ids = torch.from_numpy(np.concatenate(rows).astype(np.int64)).to(_DEV)
    last = torch.tensor(np.cumsum(spans) - 1, device=_DEV)
    if kind == "reply":
        last = torch.arange(len(g["context"]), spans[0], device=_DEV)
    V = _vocab(cfg)
    if _layered(cfg):
        x = _experts_decoder(cfg, ids, spans)[last]
        head = _streams(["head"], V * cfg["width"], cfg["width"] ** -0.5)[0].reshape(V, -1)
        logits = torch.cat([x @ part.bfloat16().double().T for part in head.split(1 << 15)], 1)
    else:
        x = (_hybrid(case, cfg, ids) if _recurrent(cfg) else _dense(case, cfg, ids, spans))[last]
        H = cfg["hidden_size"]
        if cfg["tie_word_embeddings"]:
            logits = _lin(dict(case, quant="none"), x, "model.embed_tokens.weight", V, H, 1.0)
        else:
            logits = _lin(case, x, "lm_head.weight", V, H)
    n = len(g.get("tokens", []))
    logits = (list(logits) if n > 1 else logits[0]) if kind == "reply" else logits[0] if kind == "prompt" else logits
    out = {"logits": logits[:, None] if kind == "round" else logits}
    if _steady(case):
        out["ids"] = [None] * (n if kind in ("reply", "round") else 1)
    return out
