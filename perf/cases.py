"""The work a program has this framework do, as cases that can be timed and checked one by one.

Five kinds, each through public entry points:
  layer    one decoder layer of a verify or decode step (qkv, attention, o, gate_up, down) over
           resident K/V, captured once in a HIP graph and replayed, as a serving loop does;
  head     the LM head over a step's rows and the sampler, captured the same way;
  mlp      the MLP (gate_up, down) over a prompt chunk's rows, as plain calls;
  prefill  a whole Engine.step of one prompt chunk, host planning included, with its logits.
Two shapes: "config", the 2048-wide 32/8-head model (int8 with a scale per row, or bf16), and
"limite", the reference's own 1280-wide 10/2-head model with head_dim 128 (int8 in groups of 64,
the converter's default, and in whole steps its sliding windows, value embeddings, XSA, gates
and MUDD). Weights are N(0, 0.02) as quantized by the converter; cached keys are rms-normed as
the engine leaves them.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "silicon-violetto_amd"))

from violetto import Engine  # noqa: E402
from violetto import _lib as L  # noqa: E402
from violetto import kernels as K  # noqa: E402
from violetto.model import CONFIG_SHAPE, REFERENCE_SHAPE, Extras, LayerScalars, SyntheticModel, limite_layout, rope_freq  # noqa: E402

PAGE = 16
WINDOW = 1024  # the reference model's sliding window
CHUNK = 512    # rows per prompt chunk an engine is made for
EPS = 2.0 ** -23
LAYERS = {"config": 2, "limite": 8}  # layers of a prefill case's model


def listed():
    return [
        # The smallest step end: one stream's five verified rows through the bf16 head, greedy.
        {"name": "head_1x5", "kind": "head", "shape": "config", "rows": 5, "temperature": 0.0},
        # Plain and speculative decoding's usual settings (T 0.6, top-p 0.95) over the large
        # vocabulary, one row for each of 32 streams.
        {"name": "head_limite_32", "kind": "head", "shape": "limite", "rows": 32, "temperature": 0.6},
        # The latency case: one stream, four drafts and the bonus token, 8192 tokens of context.
        {"name": "layer_1x5", "kind": "layer", "shape": "config", "fmt": "i8", "streams": 1, "rows": 5, "lo": 8192, "hi": 8192, "tree": False},
        # Plain decoding of one stream of the reference's model, an odd context.
        {"name": "layer_limite_1x1", "kind": "layer", "shape": "limite", "fmt": "g64", "streams": 1, "rows": 1, "lo": 3001, "hi": 3001, "tree": False},
        # Serving: 32 streams of uneven contexts, four drafts each.
        {"name": "layer_32x5", "kind": "layer", "shape": "config", "fmt": "i8", "streams": 32, "rows": 5, "lo": 1024, "hi": 8192, "tree": False},
        # Serving with draft trees of 16 nodes.
        {"name": "layer_32x16_tree", "kind": "layer", "shape": "config", "fmt": "i8", "streams": 32, "rows": 16, "lo": 4096, "hi": 4096, "tree": True},
        # Serving the reference's model with its drafter's blocks of 8 rows.
        {"name": "layer_limite_32x8", "kind": "layer", "shape": "limite", "fmt": "g64", "streams": 32, "rows": 8, "lo": 1024, "hi": 8192, "tree": False},
        # Long documents: 8 streams of 65536 tokens, bf16 weights.
        {"name": "layer_bf16_8x5_64k", "kind": "layer", "shape": "config", "fmt": "bf16", "streams": 8, "rows": 5, "lo": 65536, "hi": 65536, "tree": False},
        # The MLP of a large prompt batch.
        {"name": "mlp_2048", "kind": "mlp", "shape": "config", "fmt": "i8", "rows": 2048},
        # Time to first token of a short prompt: an odd number of rows, nothing cached.
        {"name": "prefill_137", "kind": "prefill", "shape": "config", "rows": 137, "ctx": 0},
        # A 512-token chunk deep in a long prompt.
        {"name": "prefill_512_32k", "kind": "prefill", "shape": "config", "rows": 512, "ctx": 32768},
        # The same of the reference's model with every layer extra, at its usual 8k.
        {"name": "prefill_limite_512_8k", "kind": "prefill", "shape": "limite", "rows": 512, "ctx": 8192},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["head", "layer", "layer", "layer", "layer", "mlp", "prefill", "prefill"])
    shape = rng.choice(["config", "config", "limite"])
    if kind == "head":
        return {"kind": kind, "shape": shape, "rows": _log(rng, 1, 32), "temperature": rng.choice([0.0, 0.6])}
    if kind == "layer":
        fmt = "g64" if shape == "limite" else rng.choice(["i8", "i8", "bf16"])
        tree = shape == "config" and rng.random() < 0.25
        streams = _log(rng, 1, 32)
        hi = _log(rng, 64, min(65536, 8 * 65536 // max(streams, 8) if fmt == "bf16" else 8192))
        lo = hi if rng.random() < 0.3 else max(1, int(hi * rng.uniform(0.1, 1.0)))
        return {"kind": kind, "shape": shape, "fmt": fmt, "streams": streams, "rows": 16 if tree else rng.randint(1, 8), "lo": lo, "hi": hi, "tree": tree}
    if kind == "mlp":
        return {"kind": kind, "shape": shape, "fmt": "g64" if shape == "limite" else rng.choice(["i8", "i8", "bf16"]), "rows": _log(rng, 17, 2048)}
    return {"kind": kind, "shape": shape, "rows": _log(rng, 17, CHUNK),
            "ctx": 0 if rng.random() < 0.3 else _log(rng, 64, 32768 if shape == "config" else 8192)}


# ------------------------------------------------------------------------------- inputs
def _shape(case):
    return CONFIG_SHAPE if case["shape"] == "config" else REFERENCE_SHAPE


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(1 + seed)
    return g


def _weight(g, m, k, fmt, std=0.02):
    """(w, scales): bf16; int8 with a bf16 scale per row ("i8") or per 64 k ("g64")."""
    w = torch.randn(m, k, generator=g, device="cuda") * std
    if fmt == "bf16":
        return w.to(torch.bfloat16), None
    w = w.view(m, 1 if fmt == "i8" else k // 64, -1)
    s = (w.abs().amax(-1) / 127).to(torch.bfloat16)
    q = (w / s.float().unsqueeze(-1)).round_().clamp_(-127, 127).to(torch.int8)
    return q.view(m, k), s


def _mats(shape):
    H, F = shape.hidden, shape.ffn
    return {"qkv": (shape.qkv_width, H), "o": (H, shape.n_heads * shape.head_dim), "gate_up": (2 * F, H), "down": (H, F)}


def _weights(g, shape, fmt, names=("qkv", "o", "gate_up", "down")):
    return {n: _weight(g, *_mats(shape)[n], fmt) for n in names}


def _mat(w):
    q, s = w
    return K.matrix(q, s, 31 if s is None or s.shape[1] == 1 else int(q.shape[1] // s.shape[1]).bit_length() - 1).tiled()


def _kv(g, layers, pages, shape):
    """K (each row of rms 1) and V of a paged cache."""
    sz = (layers, pages, shape.n_kv_heads, PAGE, shape.head_dim)
    k = torch.randn(sz, generator=g, device="cuda")
    k *= torch.rsqrt(k.square().mean(-1, keepdim=True))
    return k.to(torch.bfloat16), torch.randn(sz, generator=g, device="cuda").to(torch.bfloat16)


def _rope(pos_n, head_dim):
    th = torch.arange(pos_n, dtype=torch.float32)[:, None] * torch.from_numpy(rope_freq(500000.0, head_dim))
    return torch.stack([th.cos(), th.sin()], -1).to(torch.bfloat16).float().cuda().contiguous()


def _contexts(case):
    r = np.random.default_rng(case["streams"] * 8191 + case["hi"])
    return [int(v) for v in r.integers(case["lo"], case["hi"] + 1, case["streams"])]


def _tree(rows, tree):
    """(parent, depth) of a run's rows: a chain, or the root, 4 children, 8 grandchildren, 3 leaves."""
    parent = [max(0, i - 1) for i in range(rows)]
    if tree:
        parent = [0] + [0] * 4 + [1 + i // 2 for i in range(8)] + [5, 7, 9]
    depth = [0] * rows
    sees = [1] * rows
    for i in range(1, rows):
        depth[i] = depth[parent[i]] + 1
        sees[i] = sees[parent[i]] | 1 << i
    return depth, sees


def _split(ctxs, nkv):
    """Cached keys per attention split: the smallest that keeps the grid within 1024 workgroups."""
    for s in range(384, 3968, 128):
        if sum(-(-c // s) + 1 for c in ctxs) * nkv <= 1024:
            return s
    return 3968


def _layer_inputs(case, seed):
    sh, g = _shape(case), _gen(seed)
    ctxs = _contexts(case)
    S, R = case["streams"], case["rows"]
    n = S * R
    depth, sees = _tree(R, case["tree"])
    per = [-(-(c + R) // PAGE) for c in ctxs]
    pages = sum(per)
    perm = torch.randperm(pages, generator=g, device="cuda").to(torch.int32)
    table = torch.zeros(S, max(per), dtype=torch.int32, device="cuda")
    at = 0
    for s in range(S):
        table[s, : per[s]] = perm[at: at + per[s]]
        at += per[s]
    i = torch.arange(n)
    ctx = torch.tensor(ctxs)
    meta = torch.stack([i // R, ctx[i // R] + torch.tensor(depth)[i % R]], 1).to(torch.int32).cuda().contiguous()
    runs = torch.stack([torch.arange(S) * R, torch.full((S,), R)], 1).to(torch.int32).cuda().contiguous()
    vis = torch.tensor(sees, dtype=torch.int32).repeat(S).cuda()
    w = _weights(g, sh, case["fmt"])
    k, v = _kv(g, 1, pages, sh)
    x = torch.randn(n, sh.hidden, generator=g, device="cuda")
    return {"w": w, "k": k, "v": v, "x": x, "table": table, "meta": meta, "runs": runs, "vis": vis, "ctxs": ctxs, "depth": depth,
            "sees": sees, "rope": _rope(max(ctxs) + R + 1, sh.head_dim)}


def _scale(sh):
    return 1.0 / math.sqrt(sh.head_dim)


def _graph(call):
    """`call` captured in a HIP graph (run twice before: attributes set, code loaded)."""
    call()
    call()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        call()
    return g


def _mm_ws(ms, n):
    return K.Workspace(max(L.lib().sv_matmul_workspace_bytes(n, m.m, m.k) for m in ms))


def _prepare_layer(case, seed):
    sh, d = _shape(case), _layer_inputs(case, seed)
    n, S, R = case["streams"] * case["rows"], case["streams"], case["rows"]
    m = {k: _mat(w) for k, w in d.pop("w").items()}
    split = _split(d["ctxs"], sh.n_kv_heads)
    aa = L.AttnArgs(split, -(-max(d["ctxs"]) // split) + 1, _scale(sh) * 1.4426950408889634, 1, 0, 0, 0, 0, 0)
    kv = L.KvArgs(1, 0, 0, S, 4, d["k"].shape[1], d["table"].shape[1], 0)
    new = lambda *s: torch.zeros(*s, device="cuda")  # noqa: E731
    o = {"qkv": new(n, sh.qkv_width), "inv": new(n), "attn": new(n, sh.n_heads * sh.head_dim), "mixed": new(n, sh.hidden),
         "act": new(n, sh.ffn), "out": new(n, sh.hidden), "k": d["k"], "v": d["v"]}
    ws = _mm_ws(m.values(), n)
    wa = K.Workspace(L.lib().sv_attn_workspace_bytes(L.P(L.Shape)(sh.c()), S, aa.max_splits, R))

    def call():
        K.matmul(m["qkv"], d["x"], o["qkv"], n=n, epi=L.EPI_NORM, flags=L.FLAG_WRITE_INV, aux=o["inv"], ws=ws)
        K.attn_verify(sh, o["qkv"], d["meta"], o["k"], o["v"], d["table"], d["rope"], kv, aa, d["runs"], S, R, d["vis"], o["attn"], ws=wa)
        K.matmul(m["o"], o["attn"], o["mixed"], n=n, epi=L.EPI_RESID, ra=1.0, rb=1.0, base=d["x"], ws=ws)
        K.matmul(m["gate_up"], o["mixed"], o["act"], n=n, epi=L.EPI_SWIGLU, ws=ws)
        K.matmul(m["down"], o["act"], o["out"], n=n, epi=L.EPI_RESID, ra=1.0, rb=1.0, base=o["mixed"], ws=ws)

    return {"graph": _graph(call), "keep": (m, d, ws, wa, kv, aa), "out": o}


def _head_inputs(case, seed):
    """The embedding and hidden rows that lean on a few tokens' directions, as a trained model's
    do: at T 0.6 most of the mass lies on those tokens, the rest on the many."""
    sh, g = _shape(case), _gen(seed)
    w = (torch.randn(sh.vocab, sh.hidden, generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    pick = torch.randint(0, sh.vocab_real, (case["rows"], 6), generator=g, device="cuda")
    mix = torch.tensor([0.62, 0.55, 0.45, 0.35, 0.3, 0.2], device="cuda")
    x = torch.einsum("rjh,j->rh", w[pick].float(), mix) / 0.02
    return w, (x + 0.4 * torch.randn(case["rows"], sh.hidden, generator=g, device="cuda")) * 2.0


def _prepare_head(case, seed):
    sh, n = _shape(case), case["rows"]
    w, x = _head_inputs(case, seed)
    m = _mat((w, None))
    rows = (L.SampleRow * n)(*[L.SampleRow((7919 * i + seed) & 0xFFFFFFFF, i, 1000 + i, case["temperature"], 0.95, L.NO_TOK) for i in range(n)])
    rt = torch.frombuffer(bytearray(bytes(rows)), dtype=torch.int32).cuda()
    meta = torch.zeros(n, 2, dtype=torch.int32, device="cuda")
    o = {"logits": torch.zeros(n, sh.vocab, device="cuda"), "ids": torch.zeros(n, dtype=torch.int32, device="cuda")}
    ws = _mm_ws([m], n)

    def call():
        K.matmul(m, x, o["logits"], n=n, epi=L.EPI_HEAD, flags=L.FLAG_NORM_IN, vocab_real=sh.vocab_real, ws=ws)
        K.sample(o["logits"], rt, o["ids"], meta, n, sh.vocab)

    return {"graph": _graph(call), "keep": (m, x, rt, meta, ws), "out": o}


def _prepare_mlp(case, seed):
    sh, g, n = _shape(case), _gen(seed), case["rows"]
    m = {k: _mat(w) for k, w in _weights(g, sh, case["fmt"], ("gate_up", "down")).items()}
    x = torch.randn(n, sh.hidden, generator=g, device="cuda")
    o = {"act": torch.zeros(n, sh.ffn, device="cuda"), "out": torch.zeros(n, sh.hidden, device="cuda")}
    return {"m": m, "x": x, "n": n, "ws": _mm_ws(m.values(), n), "out": o}


def _run_mlp(s):
    o = s["out"]
    K.matmul(s["m"]["gate_up"], s["x"], o["act"], n=s["n"], epi=L.EPI_SWIGLU, ws=s["ws"])
    K.matmul(s["m"]["down"], o["act"], o["out"], n=s["n"], epi=L.EPI_RESID, ra=1.0, rb=1.0, base=s["x"], ws=s["ws"])
    return o


def _prefill_inputs(case, seed):
    """Tokens, weights, extras ("limite") and the pools: the paged layers' and the rings'."""
    sh, g = _shape(case), _gen(seed)
    nl = LAYERS[case["shape"]]
    local = limite_layout(nl)[0] if case["shape"] == "limite" else [0] * nl
    d = {"local": local, "tokens": torch.randint(0, sh.vocab_real, (case["rows"],), generator=g, device="cuda").tolist()}
    d["embed"] = (torch.randn(sh.vocab, sh.hidden, generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    d["layers"] = [_weights(g, sh, "i8" if case["shape"] == "config" else "g64") for _ in range(nl)]
    pages = -(-(case["ctx"] + case["rows"] + PAGE) // PAGE)
    d["k"], d["v"] = _kv(g, nl - sum(local), pages, sh)
    if sum(local):
        d["ring"] = -(-(WINDOW + CHUNK) // PAGE)
        d["kl"], d["vl"] = _kv(g, sum(local), d["ring"], sh)
        rn = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
        _, ve, sites, taps = limite_layout(nl)
        mix = rn(len(sites), 2, 3, 33) * 0.02
        mix[..., 32] += torch.tensor([0.1, 0.1, 1.0], device="cuda")
        d["extras"] = Extras(local, WINDOW, [rn(sh.n_heads, sh.head_dim) * 0.05 for _ in range(nl)],
                             [rn(sh.n_kv_heads, 12) * 0.3 if e else None for e in ve],
                             [torch.rand(sh.n_heads, generator=g, device="cuda") for _ in range(nl)],
                             rn(sh.vocab, sh.n_kv_heads * sh.head_dim).to(torch.bfloat16), rn(32, sh.hidden) * 0.05, mix, sites, taps)
    return d


def _model_shape(case):
    sh = _shape(case)
    return type(sh)(sh.hidden, sh.n_heads, sh.n_kv_heads, sh.head_dim, sh.ffn, sh.vocab, sh.vocab_real, LAYERS[case["shape"]])


def _prepare_prefill(case, seed):
    sh, d = _model_shape(case), _prefill_inputs(case, seed)
    total = case["ctx"] + case["rows"] + PAGE
    limite = "extras" in d
    eng = Engine(sh, max_seqs=1, max_step_tokens=CHUNK, max_seq_len=max(total, WINDOW), max_head_rows=4, kv_tokens=total, attn_scale=_scale(sh),
                 local=d["local"] if limite else None, window=WINDOW if limite else 0)
    model = SyntheticModel(sh, True, torch.device("cuda"), d["embed"], d["layers"], [LayerScalars() for _ in range(sh.n_layers)])
    if limite:
        model = model.with_extras(d["extras"])
    eng.set_model(model)
    k, v = eng.kv_cache()
    k.copy_(d["k"])
    v.copy_(d["v"])
    out = {"k": k, "v": v}
    if limite:
        kl, vl, _ = eng.local_cache()
        kl.copy_(d["kl"])
        vl.copy_(d["vl"])
        out.update(kl=kl, vl=vl)
    for t in out.values():
        t.engine = eng  # views of the engine's memory: it lives as long as they do
    torch.cuda.synchronize()
    return {"eng": eng, "ctx": case["ctx"], "tokens": d["tokens"], "out": out}


def _run_prefill(s):
    """The chunk as the next step of a sequence whose first `ctx` positions are cached."""
    eng = s["eng"]
    slot = eng.new_seq()
    if s["ctx"]:
        eng.bench_fill(slot, s["ctx"])
    r = eng.step([(slot, s["tokens"], False, 1)], logits=True)
    eng.free_seq(slot)
    return {"logits": r.logits, **s["out"]}


def prepare(case, seed):
    return {"layer": _prepare_layer, "head": _prepare_head, "mlp": _prepare_mlp, "prefill": _prepare_prefill}[case["kind"]](case, seed) | {"kind": case["kind"]}


def run(state):
    if state["kind"] == "prefill":
        return _run_prefill(state)
    if state["kind"] == "mlp":
        return _run_mlp(state)
    state["graph"].replay()
    return state["out"]


# --------------------------------------------------------------------------- work, bounds
def _bytes(fmt, m, k):
    return 2 * m * k if fmt == "bf16" else m * k + 2 * m * (1 if fmt == "i8" else k // 64)


def work(case):
    sh, n = _shape(case), case["rows"]
    H, F = sh.hidden, sh.ffn
    if case["kind"] == "head":
        return {"bytes": 2 * sh.vocab * H + 4 * n * (H + 2 * sh.vocab), "flops": 2 * n * sh.vocab * H}
    if case["kind"] == "mlp":
        mats = [_mats(sh)[k] for k in ("gate_up", "down")]
        return {"bytes": sum(_bytes(case["fmt"], *m) for m in mats) + 4 * n * (3 * H + 2 * F), "flops": 2 * n * sum(m * k for m, k in mats)}
    mats = _mats(sh).values()
    kvb = 4 * sh.n_kv_heads * sh.head_dim  # K and V of a token, bf16
    per_key = 4 * sh.n_heads * sh.head_dim  # scores and values, one query row and key
    if case["kind"] == "layer":
        ctxs = _contexts(case)
        rows, n = n, n * len(ctxs)
        keys = sum(ctxs)
        return {"bytes": sum(_bytes(case["fmt"], *m) for m in mats) + kvb * (keys + n) + 8 * n * H,
                "flops": 2 * n * sum(m * k for m, k in mats) + per_key * (rows * keys + n * (rows + 1) // 2)}
    fmt = "i8" if case["shape"] == "config" else "g64"
    by = fl = 0
    for loc in (limite_layout(LAYERS["limite"])[0] if case["shape"] == "limite" else [0] * LAYERS["config"]):
        past = min(case["ctx"], WINDOW) if loc else case["ctx"]
        by += sum(_bytes(fmt, *m) for m in mats) + kvb * (past + n)
        fl += 2 * n * sum(m * k for m, k in mats) + per_key * sum(min(i + case["ctx"], WINDOW if loc else 1 << 30) + 1 for i in range(n))
    return {"bytes": by + 2 * sh.vocab * H + 2 * n * H + 4 * sh.vocab, "flops": fl + 2 * sh.vocab * H}


def tolerance(case):
    """About four times the error against exact() (head 1e-7, mlp 3.6e-6, layer 1.3e-5 over short
    contexts); the caches of a prefill hold K and V rounded to bf16, where a last-bit change
    before the rounding moves about 0.1 % of the values by one step (1e-4 a layer, more over eight)."""
    return {"head": {"rel": 2e-6, "differ": 0.0}, "mlp": {"rel": 1.5e-5}, "layer": {"rel": 2e-4}, "prefill": {"rel": 1.5e-3}}[case["kind"]]


# ------------------------------------------------------------------------- in 64 bits
def _w64(w):
    q, s = w
    if s is None:
        return q.double()
    return (q.double().view(q.shape[0], s.shape[1], -1) * s.double().unsqueeze(-1)).view(q.shape)


def _norm(x):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)


def _rotate(x, pos, rope):
    """RoPE on the pairs (2j, 2j + 1), j < 32, of [n][heads][D] at positions pos."""
    cs = rope[pos].double().unsqueeze(1)
    a, b = x[..., 0:64:2], x[..., 1:64:2]
    y = x.clone()
    y[..., 0:64:2] = cs[..., 0] * a + cs[..., 1] * b
    y[..., 1:64:2] = cs[..., 0] * b - cs[..., 1] * a
    return y


def _heads(sh, qkv):
    n, D = qkv.shape[0], sh.head_dim
    q, k, v = qkv.split([sh.n_heads * D, sh.n_kv_heads * D, sh.n_kv_heads * D], 1)
    return q.view(n, -1, D), k.view(n, -1, D), v.view(n, -1, D)


def _attend(sh, q, keys, vals, ok):
    """softmax(q k / sqrt(D)) v of q [n][NQ][D] over keys [t][NKV][D] where ok [n][t]."""
    G = sh.n_heads // sh.n_kv_heads
    out = torch.empty_like(q)
    for h in range(sh.n_heads):
        s = q[:, h] @ keys[:, h // G].double().T.contiguous() * _scale(sh)
        out[:, h] = s.masked_fill_(~ok, -math.inf).softmax(-1) @ vals[:, h // G].double()
    return out


def _swiglu(x, w):
    gu = _norm(x) @ w.T
    return torch.nn.functional.silu(gu[:, 0::2]) * gu[:, 1::2]


def _cached(pool, pages):
    """A layer's rows in position order: pool [pages][NKV][PAGE][D] -> [t][NKV][D]."""
    return pool[pages.long()].transpose(1, 2).reshape(-1, pool.shape[1], pool.shape[3])


def _exact_layer(case, seed):
    sh, d = _shape(case), _layer_inputs(case, seed)
    R, w = case["rows"], {k: _w64(v) for k, v in d["w"].items()}
    x = d["x"].double()
    qkv = _norm(x) @ w["qkv"].T
    q, k, v = _heads(sh, qkv)
    pos = d["meta"][:, 1].long()
    q, k = _rotate(_norm(q), pos, d["rope"]), _rotate(_norm(k), pos, d["rope"]).to(torch.bfloat16)
    v = v.to(torch.bfloat16)
    sees = torch.tensor([[s >> j & 1 for j in range(R)] for s in d["sees"]], dtype=torch.bool, device="cuda")
    attn = torch.empty_like(q)
    for s, c in enumerate(d["ctxs"]):
        t = slice(s * R, s * R + R)
        pages = d["table"][s]
        keys = torch.cat([_cached(d["k"][0], pages)[:c], k[t]])
        vals = torch.cat([_cached(d["v"][0], pages)[:c], v[t]])
        attn[t] = _attend(sh, q[t], keys, vals, torch.cat([torch.ones(R, c, dtype=torch.bool, device="cuda"), sees], 1))
    attn = attn.reshape(len(x), -1)
    mixed = x + attn @ w["o"].T
    act = _swiglu(mixed, w["gate_up"])
    return {"qkv": qkv, "inv": torch.rsqrt(x.square().mean(-1) + EPS), "attn": attn, "mixed": mixed, "act": act,
            "out": mixed + act @ w["down"].T, "k": None, "v": None}


def _exact_prefill(case, seed):
    sh, d = _model_shape(case), _prefill_inputs(case, seed)
    n, ctx, NKV, D = case["rows"], case["ctx"], sh.n_kv_heads, sh.head_dim
    G = sh.n_heads // NKV
    x = d.get("extras")
    tok = torch.tensor(d["tokens"], device="cuda")
    rope = _rope(ctx + n, D)
    pos = torch.arange(ctx, ctx + n, device="cuda")
    h = h0 = _norm(d["embed"][tok].double())
    taps, glob, loc = {}, 0, 0
    for li, lw in enumerate(d["layers"]):
        w = {k: _w64(v) for k, v in lw.items()}
        a = res = h
        if x and li in x.mudd_layer:
            s = x.mudd_layer.index(li)
            inner = torch.nn.functional.gelu(_norm(h) @ x.mudd_dense1.double().T)
            m = x.mudd_mix[s].double()
            c = (inner @ m[..., :32].reshape(6, 32).T + m[..., 32].reshape(6)).unsqueeze(-1)
            a, res = (c[:, 3 * i] * h0 + c[:, 3 * i + 1] * taps[x.mudd_tap[s]] + c[:, 3 * i + 2] * h for i in (0, 1))
        xn = _norm(a)
        q, k, v = _heads(sh, xn @ w["qkv"].T)
        if x and x.ve_gate[li] is not None:
            gate = 2 * torch.sigmoid(xn[:, :12] @ x.ve_gate[li].double().T)
            v = v + gate.unsqueeze(-1) * x.value_embed[tok].double().view(n, NKV, D)
        q, k = _norm(q), _norm(k)
        if d["local"][li] or not x:
            q, k = _rotate(q, pos, rope), _rotate(k, pos, rope)
        if d["local"][li]:
            first = max(0, ctx - WINDOW) // PAGE * PAGE
            pages = torch.arange(first // PAGE, -(-ctx // PAGE), device="cuda") % d["ring"]
            kc, vc = (_cached(d[p][loc], pages)[: ctx - first] for p in ("kl", "vl"))
            loc += 1
        else:
            first = 0
            pages = torch.arange(-(-ctx // PAGE), device="cuda")
            kc, vc = (_cached(d[p][glob], pages)[:ctx] for p in ("k", "v"))
            glob += 1
        kpos = torch.cat([torch.arange(first, ctx, device="cuda"), pos])
        ok = kpos <= pos[:, None]
        if d["local"][li]:
            ok &= kpos >= pos[:, None] - WINDOW
        o = _attend(sh, q, torch.cat([kc, k.to(torch.bfloat16)]), torch.cat([vc, v.to(torch.bfloat16)]), ok)
        if x:
            vd = (v / v.norm(dim=-1, keepdim=True).clamp_min(1e-4)).repeat_interleave(G, 1)
            o = o - x.xsa[li].double()[:, None] * (o * vd).sum(-1, keepdim=True) * vd
            o = o * (2 * torch.sigmoid(xn[:, :D] @ x.attn_gate[li].double().T)).unsqueeze(-1)
        mixed = res + o.reshape(n, -1) @ w["o"].T
        h = mixed + _swiglu(mixed, w["gate_up"]) @ w["down"].T
        taps[li] = h
    lg = 23 * torch.sigmoid((_norm(h[-1:]) @ d["embed"].double().T + 5) / 7.5)
    lg[:, sh.vocab_real:] = -math.inf
    return {"logits": lg, "k": None, "v": None, **({"kl": None, "vl": None} if x else {})}


def exact(case, seed):
    if case["kind"] == "layer":
        return _exact_layer(case, seed)
    if case["kind"] == "prefill":
        return _exact_prefill(case, seed)
    sh = _shape(case)
    if case["kind"] == "head":
        w, x = _head_inputs(case, seed)
        lg = 23 * torch.sigmoid((_norm(x.double()) @ w.double().T + 5) / 7.5)
        lg[:, sh.vocab_real:] = -math.inf
        return {"logits": lg, "ids": None}
    g = _gen(seed)
    w = {k: _w64(v) for k, v in _weights(g, sh, case["fmt"], ("gate_up", "down")).items()}
    x = torch.randn(case["rows"], sh.hidden, generator=g, device="cuda").double()
    act = _swiglu(x, w["gate_up"])
    return {"act": act, "out": x + act @ w["down"].T}
