"""The work this library is measured on: the attention of its decoders' steps and prompts, the projections either side and
the IR self-attention, each through the Python entry points (dooms_amd.attention), as a decoder loop calls them.

A case is a dict of plain values. `kind` names the entry point; the other keys are its shape:

  decode          one decode step's attention on f16 query rows over per-sequence caches, one call per layer
  decode_f32      the same on f32 rows (Whisper's cross-attention over one shared encoder cache, `n_q` rows)
  decode_rope     the fused step: f32 q|k|v rows in, rotated, the new key and value appended, attended
  prefill         a prompt chunk's f16 rows against the cache, with the decoder's workspace
  prefill_rope    a prompt chunk's f32 q|k|v rows: rotated, stored into the cache, attended
  linear          a projection over f16 weights, `count` matrices a call, one call per layer
  self_attention  the IR op on packed q|k|v rows

Layers have their own caches and weights, so that a pass reads them from HBM as a decoder's step does.
"""
import math

import torch

from dooms_amd import _lib
from dooms_amd import attention as A

DEV = "cuda"

# The decoders of this repository's tests and benchmark: query heads, kv heads, head dim, rotary mode (0 adjacent pairs,
# 1 split halves, 2 none), rotary base, width, and the projections either side of the attention as (N, K).
MODELS = {
    "qwen2.5-0.5b": dict(n_head=14, n_head_kv=2, head_dim=64, rope=1, base=1e6, width=896),
    "qwen2.5-7b": dict(n_head=28, n_head_kv=4, head_dim=128, rope=1, base=1e6, width=3584),
    "llama-3-8b": dict(n_head=32, n_head_kv=8, head_dim=128, rope=0, base=5e5, width=4096),
    "whisper-large-v3-turbo": dict(n_head=20, n_head_kv=20, head_dim=64, rope=2, base=1e4, width=1280),
}
FRAMES = 1500  # encoder frames of one Whisper window


def _attn(model):
    return {k: MODELS[model][k] for k in ("n_head", "n_head_kv", "head_dim")}


def _qkv_shape(model):
    m = MODELS[model]
    return (m["n_head"] + 2 * m["n_head_kv"]) * m["head_dim"], m["width"]


def listed():
    return [
        # the smallest call: one layer's fused step of a small model at a chat-length context; latency and launch bound
        dict(name="step_qwen05b_513", kind="decode_rope", model="qwen2.5-0.5b", batch=1, kv_min=513, kv_max=513, layers=1),
        # a single user's long context: the attention of eight layers of one step, each over 8192 keys of its own
        dict(name="decode_llama8b_8192", kind="decode", model="llama-3-8b", batch=1, kv_min=8192, kv_max=8192, n_q=1, layers=8),
        # a serving step: sixteen sequences of very different lengths, one layer, the fused step
        dict(name="step_llama8b_batch16", kind="decode_rope", model="llama-3-8b", batch=16, kv_min=1025, kv_max=8191, layers=1),
        # Whisper beam search: the four decoder layers' cross-attention of one token, five beams over one encoder cache
        dict(name="cross_whisper_beam5", kind="decode_f32", model="whisper-large-v3-turbo", batch=1, kv_min=FRAMES, kv_max=FRAMES, n_q=5, layers=4),
        # a short prompt, whole: time to first token of a small model
        dict(name="prompt_qwen05b_512", kind="prefill_rope", model="qwen2.5-0.5b", n_q=512, p0=0),
        # a long prompt, whole, of an odd length
        dict(name="prompt_llama8b_3999", kind="prefill_rope", model="llama-3-8b", n_q=3999, p0=0),
        # the last chunk of a 32k prompt taken 2048 rows at a time: the largest call
        dict(name="chunk_qwen7b_32k", kind="prefill", model="qwen2.5-7b", n_q=2048, p0=30720),
        # a single user's token through the normalized q|k|v projection of eight layers: bound by the weights
        dict(name="qkv_llama8b_1", kind="linear", n=6144, k=4096, m=1, count=1, layers=8, norm=True, accumulate=False, bias=False, f16=False),
        # a serving step's 24 rows through the output projection into the residual, four layers
        dict(name="out_llama8b_24", kind="linear", n=4096, k=4096, m=24, count=1, layers=4, norm=False, accumulate=True, bias=False, f16=False),
        # a prompt chunk through the normalized q|k|v projection
        dict(name="qkv_llama8b_2048", kind="linear", n=6144, k=4096, m=2048, count=1, layers=1, norm=True, accumulate=False, bias=False, f16=False),
        # one audio window's keys and values for Whisper's four cross-attention layers, straight into the f16 caches
        dict(name="cross_cache_whisper", kind="linear", n=1280, k=1280, m=FRAMES, count=8, layers=1, norm=False, accumulate=False, bias=True, f16=True),
        # an image encoder's layer: four images of 1024 patches, bf16
        dict(name="vit_l_4x1024_bf16", kind="self_attention", batch=4, n=1024, heads=16, head_dim=64, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed kinds: any decoder, lengths and row counts over their whole range."""
    while True:
        c = _draw(rng)
        w = work(c)
        if w["flops"] <= 0.96e12 and w["bytes"] <= 0.6e9 and w["flops"] / 8e14 + w["bytes"] / 5e12 < 1.1e-3:
            return c


def _draw(rng):
    kind = rng.choice(["decode", "decode_f32", "decode_rope", "prefill", "prefill_rope", "linear", "linear", "linear", "self_attention"])
    llms = ["qwen2.5-0.5b", "qwen2.5-7b", "llama-3-8b"]
    if kind in ("decode", "decode_rope"):
        model = rng.choice(llms + ["whisper-large-v3-turbo"])
        top = 448 if model.startswith("whisper") else 16384  # Whisper's text context
        hi = _log(rng, 16, top)
        c = dict(kind=kind, model=model, batch=rng.choice([1, 1, 2, 3, 4, 5, 8, 16]), kv_min=rng.randint(max(1, hi // 8), hi), kv_max=hi,
                 layers=rng.choice([1, 2, 4]))
        return dict(c, n_q=1) if kind == "decode" else c
    if kind == "decode_f32":
        frames = rng.choice([FRAMES, FRAMES, rng.randint(100, FRAMES)])
        return dict(kind=kind, model="whisper-large-v3-turbo", batch=rng.choice([1, 1, 4]), kv_min=frames, kv_max=frames, n_q=rng.randint(1, 8), layers=4)
    if kind in ("prefill", "prefill_rope"):
        model = rng.choice(llms)
        n_q = _log(rng, 16, 4096)
        return dict(kind=kind, model=model, n_q=n_q, p0=rng.choice([0, 0, n_q, _log(rng, 64, 30720)]))
    if kind == "linear":
        m = _log(rng, 1, 4096)
        if 8 < m <= 16:  # a version of the library read ahead of its workspace at these row counts: not timed
            m += 8
        model = rng.choice(llms + ["whisper-large-v3-turbo"])
        w = MODELS[model]["width"]
        if model.startswith("whisper") and m > 256:
            return dict(kind=kind, n=w, k=w, m=m, count=8, layers=1, norm=False, accumulate=False, bias=True, f16=True)
        layers = 4 if m <= 64 else 1
        if rng.random() < 0.5:
            n, k = _qkv_shape(model)
            return dict(kind=kind, n=n, k=k, m=m, count=1, layers=layers, norm=True, accumulate=False, bias=model.startswith("qwen"), f16=False)
        if model == "llama-3-8b" and rng.random() < 0.4:  # the feed-forward's down projection
            return dict(kind=kind, n=w, k=14336, m=m, count=1, layers=layers, norm=False, accumulate=True, bias=False, f16=False)
        return dict(kind=kind, n=w, k=w, m=m, count=1, layers=layers, norm=False, accumulate=True, bias=False, f16=False)
    heads, head_dim = rng.choice([(12, 64), (16, 64), (16, 80), (16, 80), (20, 64)])
    return dict(kind=kind, batch=rng.choice([1, 2, 4, 8]), n=rng.randint(50, 1500), heads=heads, head_dim=head_dim, dtype=rng.choice(["f32", "f16", "bf16"]))


def _lens(c):
    """The sequences' lengths, spread evenly from the longest down to the shortest."""
    b, lo, hi = c["batch"], c["kv_min"], c["kv_max"]
    return [hi - (hi - lo) * i // max(1, b - 1) for i in range(b)]


class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)

    def __call__(self, *shape, dtype=torch.float16, std=1.0):
        x = torch.randn(*shape, generator=self.g, device=DEV, dtype=torch.float32)
        return (x * std if std != 1.0 else x).to(dtype)


def _inputs(c, seed):
    """The tensors a decoder holds before the call, from the seed alone."""
    r, kind = _Rand(seed), c["kind"]
    f32 = torch.float32
    s = {}
    if kind.startswith("decode"):
        m = MODELS[c["model"]]
        qw, kw = m["n_head"] * m["head_dim"], m["n_head_kv"] * m["head_dim"]
        lens, rows = _lens(c), c["batch"] * c.get("n_q", 1)
        s["k"] = [[r(n, kw) for n in lens] for _ in range(c["layers"])]
        s["v"] = [[r(n, kw) for n in lens] for _ in range(c["layers"])]
        w, dt = (qw + 2 * kw, f32) if kind == "decode_rope" else (qw, f32 if kind == "decode_f32" else torch.float16)
        s["q"] = [r(rows, w, dtype=dt) for _ in range(c["layers"])]
    elif kind.startswith("prefill"):
        m = MODELS[c["model"]]
        qw, kw = m["n_head"] * m["head_dim"], m["n_head_kv"] * m["head_dim"]
        n_kv = c["p0"] + c["n_q"]
        s["k"], s["v"] = r(n_kv, kw, std=0.5 ** 0.5), r(n_kv, kw, std=0.5 ** 0.5)
        if kind == "prefill":
            s["q"] = r(c["n_q"], qw, std=0.5 ** 0.5)
        else:
            s["q"] = r(c["n_q"], qw + 2 * kw, dtype=f32)
    elif kind == "linear":
        M, N, K = c["m"], c["n"], c["k"]
        s["x"] = [r(M, K, dtype=f32) for _ in range(c["layers"])]
        s["w"] = [[r(N, K, std=K ** -0.5) for _ in range(c["count"])] for _ in range(c["layers"])]
        s["gamma"] = [1 + r(K, dtype=f32, std=0.1) if c["norm"] else None for _ in range(c["layers"])]
        s["bias"] = [[r(N, dtype=f32, std=0.1) for _ in range(c["count"])] if c["bias"] else None for _ in range(c["layers"])]
        s["y"] = [[r(M, N, dtype=f32) if c["accumulate"] else torch.empty(M, N, device=DEV, dtype=torch.float16 if c["f16"] else f32)
                   for _ in range(c["count"])] for _ in range(c["layers"])]
    else:
        dt = dict(f32=torch.float32, f16=torch.float16, bf16=torch.bfloat16)[c["dtype"]]
        s["qkv"] = r(c["batch"], c["n"], 3 * c["heads"] * c["head_dim"], dtype=dt)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    kind = s["kind"] = case["kind"]
    if kind.startswith("decode"):
        s["args"] = _attn(case["model"])
        s["lens"] = _lens(case)
        n_q = case.get("n_q", 1)
        need = A.decode_workspace_bytes(**s["args"], n_q=n_q, batch=case["batch"], max_kv_len=max(s["lens"]))
        s["ws"] = A.new_workspace(need, torch.device(DEV))
        if kind == "decode_rope":
            m = MODELS[case["model"]]
            s["args"].update(rope_mode=m["rope"], rope_base=m["base"])
        else:
            s["args"].update(n_q=n_q)
    elif kind.startswith("prefill"):
        m, rope = MODELS[case["model"]], kind == "prefill_rope"
        s["args"] = dict(_attn(case["model"]), p0=case["p0"])
        qw, kw = m["n_head"] * m["head_dim"], m["n_head_kv"] * m["head_dim"]
        d = _lib.make_desc(m["n_head"], m["n_head_kv"], m["head_dim"], case["n_q"], s["q"].stride(0), kw, qw,
                           1 / math.sqrt(m["head_dim"]), p0=case["p0"])
        s["ws"] = A.new_workspace(_lib.prefill_workspace_bytes(d), torch.device(DEV))
        if rope:
            s["args"].update(rope_mode=m["rope"], rope_base=m["base"])
            s["rows"] = slice(case["p0"], case["p0"] + case["n_q"])
    elif kind == "linear":
        s["args"] = dict(accumulate=case["accumulate"], out_f16=case["f16"])
    else:
        s["heads"] = case["heads"]
    return s


def run(s):
    kind = s["kind"]
    if kind in ("decode", "decode_f32"):
        return [A.decode(q, k, v, s["lens"], workspace=s["ws"], **s["args"])[0] for q, k, v in zip(s["q"], s["k"], s["v"])]
    if kind == "decode_rope":
        out = [A.decode_rope(q, k, v, s["lens"], workspace=s["ws"], **s["args"])[0] for q, k, v in zip(s["q"], s["k"], s["v"])]
        # the appended rows are each cache's last
        return {"out": out, "k": s["k"][0][0][-1], "v": s["v"][0][0][-1]}
    if kind == "prefill":
        return A.prefill(s["q"], s["k"], s["v"], workspace=s["ws"], want_lse=True, **s["args"])
    if kind == "prefill_rope":
        out, _ = A.prefill_rope(s["q"], s["k"], s["v"], workspace=s["ws"], **s["args"])
        return {"out": out, "k": s["k"][s["rows"]], "v": s["v"][s["rows"]]}
    if kind == "linear":
        return [A.linear(x, w, out=y, gamma=g, bias=b, **s["args"]) for x, w, y, g, b in zip(s["x"], s["w"], s["y"], s["gamma"], s["bias"])]
    return A.self_attention(s["qkv"], heads=s["heads"])


def work(case):
    """Each input read once, each output written once; two operations per multiply-add, visible (query, key) pairs only."""
    kind = case["kind"]
    if kind.startswith("decode"):
        m, n_q = MODELS[case["model"]], case.get("n_q", 1)
        qw, kw = m["n_head"] * m["head_dim"], m["n_head_kv"] * m["head_dim"]
        keys, rows = sum(_lens(case)), case["batch"] * n_q
        es = 2 if kind == "decode" else 4
        b = keys * kw * 2 * 2 + rows * qw * 2 * es + (rows * 2 * kw * 4 if kind == "decode_rope" else 0)
        return {"bytes": case["layers"] * b, "flops": case["layers"] * 4 * qw * keys * n_q}
    if kind.startswith("prefill"):
        m, n_q, p0 = MODELS[case["model"]], case["n_q"], case["p0"]
        qw, kw = m["n_head"] * m["head_dim"], m["n_head_kv"] * m["head_dim"]
        pairs = n_q * p0 + n_q * (n_q + 1) // 2
        if kind == "prefill":
            b = n_q * qw * 2 * 2 + (p0 + n_q) * kw * 2 * 2 + n_q * m["n_head"] * 4
        else:
            b = n_q * (qw + 2 * kw) * 4 + n_q * qw * 4 + (p0 + n_q) * kw * 2 * 2
        return {"bytes": b, "flops": 4 * qw * pairs}
    if kind == "linear":
        M, N, K, n = case["m"], case["n"], case["k"], case["count"]
        y = M * N * (2 if case["f16"] else 8 if case["accumulate"] else 4)
        return {"bytes": case["layers"] * (M * K * 4 + n * (N * K * 2 + y)), "flops": case["layers"] * n * 2 * M * N * K}
    B, N, E = case["batch"], case["n"], case["heads"] * case["head_dim"]
    return {"bytes": 4 * B * N * E * (4 if case["dtype"] == "f32" else 2), "flops": 4 * B * N * N * E}


def tolerance(case):
    """About four times the largest error against exact() that the case's kind shows: the operands' rounding to half (and
    bf16's output), or f32 sums for the projections of few rows."""
    kind = case["kind"]
    if kind == "linear":
        if case["m"] <= 8 and not case["f16"]:
            return {"rel": 1e-5}
        return {"rel": 1.5e-3}
    if kind == "self_attention":
        return {"rel": 1e-2 if case["dtype"] == "bf16" else 2.5e-3}
    return {"rel": 2.5e-3}


def _softmax_v(q, k, v, visible):
    """softmax(q k^T / sqrt(d)) v and the log-sum-exp, in 64 bits, rows in blocks: q [rows][d], k and v [keys][d];
    row i sees keys 0 .. visible[i] - 1."""
    out, lse = [], []
    step = max(1, (1 << 27) // k.shape[0])
    pos = torch.arange(k.shape[0], device=q.device)
    for i in range(0, q.shape[0], step):
        s = q[i:i + step] @ k.T / math.sqrt(q.shape[1])
        s.masked_fill_(pos[None, :] >= visible[i:i + step, None], -math.inf)
        lse.append(torch.logsumexp(s, 1))
        out.append(torch.softmax(s, 1) @ v)
    return torch.cat(out), torch.cat(lse)


def _rotate(x, heads, hd, pos, mode, base):
    """Rotary embedding of x [rows][heads hd] at positions pos, in 64 bits, at the f32 angles float(pos) * f32 frequency."""
    x = x.double().view(-1, heads, hd)
    if mode == 2:
        return x
    freq = (base ** (-2 * torch.arange(hd // 2, device=x.device, dtype=torch.float64) / hd)).float()
    ang = (pos.float()[:, None] * freq[None, :]).double()[:, None, :]
    c, s = ang.cos(), ang.sin()
    a, b = (x[..., 0::2], x[..., 1::2]) if mode == 0 else (x[..., :hd // 2], x[..., hd // 2:])
    ra, rb = a * c - b * s, a * s + b * c
    return torch.stack((ra, rb), -1).flatten(2) if mode == 0 else torch.cat((ra, rb), -1)


def _attend(q, k, v, visible):
    """q [rows][heads][d], k and v [keys][kv heads][d] in 64 bits: out [rows][heads d], lse [rows][heads]."""
    g = q.shape[1] // k.shape[1]
    both = [_softmax_v(q[:, h], k[:, h // g], v[:, h // g], visible) for h in range(q.shape[1])]
    return torch.stack([o for o, _ in both], 1).flatten(1), torch.stack([l for _, l in both], 1)


def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind.startswith("decode"):
        m = MODELS[case["model"]]
        H, G, d = m["n_head"], m["n_head_kv"], m["head_dim"]
        lens, n_q = _lens(case), case.get("n_q", 1)
        outs, first = [], None
        for layer in range(case["layers"]):
            rows = []
            for b, n in enumerate(lens):
                q = s["q"][layer][b * n_q:(b + 1) * n_q].double()
                k, v = s["k"][layer][b].double().view(n, G, d), s["v"][layer][b].double().view(n, G, d)
                if kind == "decode_rope":
                    pos = torch.tensor([n - 1], device=DEV)
                    k[-1] = _rotate(q[:, H * d:(H + G) * d], G, d, pos, m["rope"], m["base"])[0]
                    v[-1] = q[0, (H + G) * d:].view(G, d)
                    first = first or (k[-1].flatten(), v[-1].flatten())
                    q = _rotate(q[:, :H * d], H, d, pos, m["rope"], m["base"])
                rows.append(_attend(q.reshape(-1, H, d), k, v, torch.full((n_q,), n, device=DEV))[0])
            outs.append(torch.cat(rows))
        return {"out": outs, "k": first[0], "v": first[1]} if kind == "decode_rope" else outs
    if kind.startswith("prefill"):
        m, n_q, p0 = MODELS[case["model"]], case["n_q"], case["p0"]
        H, G, d = m["n_head"], m["n_head_kv"], m["head_dim"]
        pos = p0 + torch.arange(n_q, device=DEV)
        k, v = s["k"].double().view(-1, G, d), s["v"].double().view(-1, G, d)
        q = s["q"].double()
        if kind == "prefill":
            return _attend(q.view(-1, H, d), k, v, pos + 1)
        k[p0:] = _rotate(q[:, H * d:(H + G) * d], G, d, pos, m["rope"], m["base"])
        v[p0:] = q[:, (H + G) * d:].reshape(-1, G, d)
        out, _ = _attend(_rotate(q[:, :H * d], H, d, pos, m["rope"], m["base"]), k, v, pos + 1)
        return {"out": out, "k": k[p0:].flatten(1), "v": v[p0:].flatten(1)}
    if kind == "linear":
        outs = []
        for x, ws, g, bs, ys in zip(s["x"], s["w"], s["gamma"], s["bias"], s["y"]):
            x = x.double()
            if g is not None:
                x = x * g.double() / (x.square().mean(1, keepdim=True) + 1e-5).sqrt()
            y = [x @ w.double().T for w in ws]
            if bs is not None:
                y = [a + b.double() for a, b in zip(y, bs)]
            if case["accumulate"]:
                y = [a + b.double() for a, b in zip(y, ys)]
            outs.append(y)
        return outs
    B, N, H, d = case["batch"], case["n"], case["heads"], case["head_dim"]
    x = s["qkv"].double().view(B, N, 3, H, d)
    return torch.stack([_attend(x[b, :, 0], x[b, :, 1], x[b, :, 2], torch.full((N,), N, device=DEV))[0] for b in range(B)])
