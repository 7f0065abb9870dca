"""What a user of this framework has it do, as cases that can be timed and compared.

Whole calls on an engine (prompt to first token, greedy generation, a sampled chat turn), and the single
operators and layers that a host program drives one by one: an attention layer, a feed-forward layer, the
greedy LM head, one matmul, one sampling step.  Two models, both named by the tests and the benchmark: the
2.4B-shaped decoder (40 layers, hidden 2304, 32/8 heads of 64, FFN 5760) and the reference file's geometry
(42 layers, hidden 2048, 16/2 heads of 128, FFN 6144); both have 130,560 tokens.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "minicpm5.cpp_amd", "python"))
import mcpm  # noqa: E402

VOCAB = 130560
# layers, hidden, heads, kv heads, head_dim, ffn, RoPE base, synthetic file layout (0: tied Q6_K embedding,
# Q6_K v and down; 2: the reference file's own mix, untied Q6_K head)
MODELS = {
    "2.4b": (40, 2304, 32, 8, 64, 5760, 1e4, 0),
    "ref": (42, 2048, 16, 2, 128, 6144, 5e6, 2),
}
WEIGHT_SEED = 20260105
MAX_SEQ = 4096  # the KV capacity an engine is opened with
EPS = 1e-6
BLOCK_BYTES = {"q4_K": (144, 256), "q6_K": (210, 256), "q8_0": (34, 32), "f32": (4, 1)}
TYPES = {"q4_K": mcpm.TYPE_Q4_K, "q6_K": mcpm.TYPE_Q6_K, "q8_0": mcpm.TYPE_Q8_0, "f32": mcpm.TYPE_F32}


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # the headline: a short prompt, then greedy tokens one by one
        dict(name="greedy_2.4b", kind="greedy", model="2.4b", prompt=32, gen=20),
        # the same on the geometry of the file that the reference ships for
        dict(name="greedy_ref", kind="greedy", model="ref", prompt=24, gen=16),
        # a long prompt up to its first token (the long-context benchmark's prompt)
        dict(name="prompt_1024", kind="first_token", model="2.4b", prompt=1024),
        # an ordinary question, a ragged length, up to its first token
        dict(name="prompt_45", kind="first_token", model="2.4b", prompt=45),
        dict(name="prompt_ref_333", kind="first_token", model="ref", prompt=333),
        # the next turn of a chat: 1500 positions already cached, 77 new tokens, sampled answer tokens
        dict(name="turn_sampled", kind="turn", model="2.4b", pos0=1500, new=77, gen=12, temperature=0.8, top_p=0.95),
        # one attention layer driven operator by operator, as a host program linked against the operators does
        dict(name="attention_513", kind="attention", model="2.4b", context=513),
        dict(name="attention_ref_4000", kind="attention", model="ref", context=4000),
        # one feed-forward layer, the same way
        dict(name="mlp", kind="mlp", model="2.4b"),
        # final norm, LM head and argmax of a greedy step
        dict(name="head", kind="head", model="2.4b"),
        # the smallest call, bound by its launch: one layer's O projection
        dict(name="matmul_o_proj", kind="matmul", type="q4_K", rows=2304, cols=2048),
        # a model kept in Q8_0: one FFN-sized matrix
        dict(name="matmul_q8_0", kind="matmul", type="q8_0", rows=2304, cols=5760),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    model = rng.choice(sorted(MODELS))
    kind = rng.choice(["greedy", "first_token", "first_token", "turn", "attention", "attention", "mlp", "matmul",
                       "matmul", "sample"])
    if kind == "greedy":
        return dict(kind=kind, model=model, prompt=_log_int(rng, 2, 200), gen=rng.randint(4, 16))
    if kind == "first_token":
        return dict(kind=kind, model=model, prompt=_log_int(rng, 2, 900))
    if kind == "turn":
        return dict(kind=kind, model=model, pos0=_log_int(rng, 100, 3000), new=_log_int(rng, 4, 150),
                    gen=rng.randint(3, 10), temperature=round(rng.uniform(0.5, 1.1), 2),
                    top_p=round(rng.uniform(0.8, 0.99), 2))
    if kind == "attention":
        return dict(kind=kind, model=model, context=_log_int(rng, 1, 4096))
    if kind == "mlp":
        # any FFN width whose blocks are whole
        return dict(kind=kind, model=model, ffn=256 * rng.randint(4, 30))
    if kind == "matmul":
        t = rng.choice(["q4_K", "q6_K", "q8_0", "f32"])
        return dict(kind=kind, type=t, rows=_log_int(rng, 1000, 8192), cols=256 * _log_int(rng, 4, 24))
    return dict(kind=kind, n=_log_int(rng, 1000, VOCAB), temperature=round(rng.uniform(0.5, 1.2), 2),
                top_p=round(rng.uniform(0.7, 0.99), 2))


# ---------------------------------------------------- weights, context, engines

_ctx = None
_images = {}
_engines = {}


def _context():
    global _ctx
    if _ctx is None:
        _ctx = mcpm.Context(0)
    return _ctx


def _engine(model, role):
    """The engine a server keeps for its life: its weights are the model's, whatever the request.  Chat turns
    have an engine of their own, whose cache holds the document that every turn continues."""
    if (model, role) not in _engines:
        if model not in _images:
            L, dim, nh, nkv, hd, ffn, base, mix = MODELS[model]
            cfg = mcpm.make_config(L, dim, nh, nkv, hd, ffn, VOCAB, rope_base=base, eps=EPS)
            _images[model] = mcpm.synth_gguf(cfg, WEIGHT_SEED, mix)
        e = mcpm.Engine(_context(), image=_images[model])
        e.init_kv_cache(MAX_SEQ)
        _engines[model, role] = e
    return _engines[model, role]


def _q4k_parts(rng, rows, cols):
    n = rows * (cols // 256)
    sc = rng.integers(20, 64, (n, 8), dtype=np.uint8)
    qs = rng.integers(0, 256, (n, 128), dtype=np.uint8)
    # d*sc*q - dmin*mn with mn = sc and dmin = 7.5 d: symmetric weights of about N(0, 0.02)'s spread
    d = rng.uniform(0.7e-4, 1.4e-4, n).astype(np.float16)
    dmin = (7.5 * d.astype(np.float32)).astype(np.float16)
    return d, dmin, sc, qs


def _q4k_blocks(parts):
    d, dmin, sc, qs = parts
    b = np.zeros(d.size, mcpm.Q4_K)
    b["d"], b["dmin"], b["qs"] = d.view(np.uint16), dmin.view(np.uint16), qs
    lo, hi = sc[:, :4], sc[:, 4:]
    top = lo | ((hi >> 4) << 6)
    b["scales"] = np.concatenate([top, top, (hi & 15) | ((hi & 15) << 4)], axis=1)
    return b


def _q4k_values(parts, rows, cols):
    d, dmin, sc, qs = (torch.from_numpy(p).cuda() for p in parts)
    q = torch.stack([qs.view(-1, 4, 32) & 15, qs.view(-1, 4, 32) >> 4], dim=2).view(-1, 8, 32).double()
    s = sc.double()[:, :, None]
    return (d.double()[:, None, None] * s * q - dmin.double()[:, None, None] * s).view(rows, cols)


def _q6k_parts(rng, rows, cols):
    n = rows * (cols // 256)
    sc = rng.integers(32, 128, (n, 16), dtype=np.int8) * rng.choice(np.array([-1, 1], np.int8), (n, 16))
    ql = rng.integers(0, 256, (n, 128), dtype=np.uint8)
    qh = rng.integers(0, 256, (n, 64), dtype=np.uint8)
    d = rng.uniform(1.0e-5, 1.8e-5, n).astype(np.float16)
    return d, sc, ql, qh


def _q6k_blocks(parts):
    d, sc, ql, qh = parts
    b = np.zeros(d.size, mcpm.Q6_K)
    b["d"], b["scales"], b["ql"], b["qh"] = d.view(np.uint16), sc, ql, qh
    return b


def _q6k_values(parts, rows, cols):
    d, sc, ql, qh = (torch.from_numpy(p).cuda() for p in parts)
    l, h = ql.view(-1, 2, 2, 32), qh.view(-1, 2, 32)
    q = torch.stack([(l[:, :, 0] & 15) | ((h & 3) << 4), (l[:, :, 1] & 15) | (((h >> 2) & 3) << 4),
                     (l[:, :, 0] >> 4) | (((h >> 4) & 3) << 4), (l[:, :, 1] >> 4) | ((h >> 6) << 4)], dim=2)
    q = q.view(-1, 16, 16).double() - 32
    return (d.double()[:, None, None] * sc.double()[:, :, None] * q).view(rows, cols)


def _q80_parts(rng, rows, cols):
    n = rows * (cols // 32)
    return rng.uniform(1.5e-4, 4e-4, n).astype(np.float16), rng.integers(-127, 128, (n, 32), dtype=np.int8)


def _parts(rng, kind, rows, cols):
    if kind == "q4_K":
        return _q4k_parts(rng, rows, cols)
    if kind == "q6_K":
        return _q6k_parts(rng, rows, cols)
    if kind == "q8_0":
        return _q80_parts(rng, rows, cols)
    return (rng.standard_normal((rows, cols), dtype=np.float32) * np.float32(0.02),)


def _upload(kind, parts, rows, cols):
    if kind == "q4_K":
        native = _q4k_blocks(parts)
    elif kind == "q6_K":
        native = _q6k_blocks(parts)
    elif kind == "q8_0":
        native = np.zeros(parts[0].size, mcpm.Q8_0)
        native["d"], native["qs"] = parts[0].view(np.uint16), parts[1]
    else:
        native = parts[0]
    return _context().tensor(native, TYPES[kind], cols, rows)


def _values(kind, parts, rows, cols):
    """The weights in 64 bits, [rows, cols]."""
    if kind == "q4_K":
        return _q4k_values(parts, rows, cols)
    if kind == "q6_K":
        return _q6k_values(parts, rows, cols)
    if kind == "q8_0":
        return (torch.from_numpy(parts[0]).cuda().double()[:, None] * torch.from_numpy(parts[1]).cuda().double()).view(rows, cols)
    return torch.from_numpy(parts[0]).cuda().double()


def _gain(rng, n):
    return (1.0 + 0.1 * rng.standard_normal(n)).astype(np.float32)


def _matrices(case):
    """name -> (type, rows, cols) of a case's weights."""
    if case["kind"] == "matmul":
        return {"w": (case["type"], case["rows"], case["cols"])}
    L, dim, nh, nkv, hd, ffn, base, mix = MODELS[case["model"]]
    if case["kind"] == "attention":
        return {"wq": ("q4_K", nh * hd, dim), "wk": ("q4_K", nkv * hd, dim), "wv": ("q6_K", nkv * hd, dim),
                "wo": ("q4_K", dim, nh * hd)}
    if case["kind"] == "mlp":
        f = case.get("ffn") or (ffn + 255) // 256 * 256
        return {"wg": ("q4_K", f, dim), "wu": ("q4_K", f, dim), "wd": ("q6_K", dim, f)}
    return {"w": ("q6_K", VOCAB, dim)}  # head


def _inputs(case, seed):
    """A single-layer case's inputs on the host: weights' parts and activations, from the seed alone."""
    rng = np.random.Generator(np.random.SFC64(seed))
    h = {"parts": {k: _parts(rng, *m) for k, m in _matrices(case).items()} if case["kind"] != "sample" else {}}
    if case["kind"] == "matmul":
        h["x"] = rng.standard_normal(case["cols"], dtype=np.float32)
    elif case["kind"] == "sample":
        h["x"] = rng.standard_normal(case["n"], dtype=np.float32) * np.float32(2.5)
        h["r"] = float(rng.uniform(0.02, 0.98))
    else:
        dim = MODELS[case["model"]][1]
        h["x"] = rng.standard_normal(dim, dtype=np.float32)
        h["gamma"] = _gain(rng, dim)
        if case["kind"] == "attention":
            _, _, nh, nkv, hd, *_ = MODELS[case["model"]]
            for k in ("k_cache", "v_cache"):
                h[k] = rng.standard_normal((_rows(case), nkv * hd), dtype=np.float32)
    return h


def _rows(case):
    """KV rows a host program holds for an attention case: whole chunks past the context."""
    return min(MAX_SEQ, (case["context"] + 511) // 512 * 512)


# ---------------------------------------------------------------- prepare, run

def _tokens(seed, n):
    return np.random.default_rng(seed).integers(0, VOCAB, n).astype(np.int32)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("greedy", "first_token"):
        return {"case": case, "engine": _engine(case["model"], "chat"), "tokens": _tokens(seed, case["prompt"])}
    if kind == "turn":
        e = _engine(case["model"], "turns")
        # the document every turn continues; its rows stay, a turn writes only those after it
        e.prefill(_tokens(WEIGHT_SEED, MAX_SEQ)[:case["pos0"]], 0)
        return {"case": case, "engine": e, "tokens": _tokens(seed, case["new"]), "seed": int(seed) & 0x7fffffff}
    h = _inputs(case, seed)
    s = {"case": case, "ctx": _context(), "x": torch.from_numpy(h["x"]).cuda()}
    dev = dict(device="cuda", dtype=torch.float32)
    if kind == "sample":
        s["r"], s["token"] = h["r"], torch.zeros(1, dtype=torch.int32, device="cuda")
    elif kind == "matmul":
        s["out"] = torch.zeros(case["rows"], **dev)
    else:
        L, dim, nh, nkv, hd, ffn, base, mix = MODELS[case["model"]]
        s["gamma"] = torch.from_numpy(h["gamma"]).cuda()
        s["xq"] = torch.zeros(dim // 256 * 292, device="cuda", dtype=torch.uint8)
        if kind == "attention":
            s["k_cache"], s["v_cache"] = (torch.from_numpy(h[k]).cuda() for k in ("k_cache", "v_cache"))
            s["q"], s["att"] = torch.zeros(nh * hd, **dev), torch.zeros(nh * hd, **dev)
            s["k"], s["v"] = torch.zeros(nkv * hd, **dev), torch.zeros(nkv * hd, **dev)
            s["out"] = torch.zeros(dim, **dev)
        elif kind == "mlp":
            f = _matrices(case)["wg"][1]
            s["gate"], s["up"] = torch.zeros(f, **dev), torch.zeros(f, **dev)
            s["hq"] = torch.zeros(f // 256 * 292, device="cuda", dtype=torch.uint8)
            s["out"] = torch.zeros(dim, **dev)
        else:
            s["norm"], s["logits"] = torch.zeros(dim, **dev), torch.zeros(VOCAB, **dev)
            s["token"] = torch.zeros(1, dtype=torch.int32, device="cuda")
    for k, m in (_matrices(case) if kind != "sample" else {}).items():
        s[k] = _upload(m[0], h["parts"][k], m[1], m[2])
    torch.cuda.synchronize()
    return s


def _run_greedy(s):
    e, t, n = s["engine"], s["tokens"], s["case"]["gen"]
    out = e.generate_greedy(t, n)
    logits, _ = e.forward(int(out[-1]), t.size + n - 1)
    return {"tokens": out, "logits": logits}


def _run_first_token(s):
    e, t = s["engine"], s["tokens"]
    e.prefill(t[:-1], 0)
    logits, token = e.forward(int(t[-1]), t.size - 1)
    return {"token": token, "logits": logits}


def _run_turn(s):
    c, e, t = s["case"], s["engine"], s["tokens"]
    out = e.generate_sampled_at(t, c["pos0"], c["gen"], c["temperature"], c["top_p"], s["seed"])
    logits, _ = e.forward(int(out[-1]), c["pos0"] + t.size + c["gen"] - 1)
    return {"tokens": out, "logits": logits}


def _run_attention(s):
    c, ctx, lib, ok = s["case"], s["ctx"].h, s["ctx"].lib, mcpm.check
    L, dim, nh, nkv, hd, ffn, base, mix = MODELS[c["model"]]
    x, gamma, xq, q, k, v, att, out, kc, vc = (s[n].data_ptr() for n in (
        "x", "gamma", "xq", "q", "k", "v", "att", "out", "k_cache", "v_cache"))
    pos = c["context"] - 1
    ok(lib.mcpm_rmsnorm_and_quantize_q8k(ctx, xq, x, gamma, dim, EPS))
    ok(lib.mcpm_gemv_qkv_q8_K(ctx, s["wq"].h, s["wk"].h, s["wv"].h, xq, q, k, v, nh * hd, nkv * hd, dim))
    ok(lib.mcpm_apply_rope(ctx, q, pos, nh, hd, base))
    ok(lib.mcpm_apply_rope(ctx, k, pos, nkv, hd, base))
    ok(lib.mcpm_execute_attention(ctx, att, q, k, v, kc, vc, pos, s["k_cache"].shape[0], nh, nkv, hd))
    ok(lib.mcpm_matmul(ctx, s["wo"].h, att, out))
    return {"attention": s["att"], "out": s["out"], "k_cache": s["k_cache"], "v_cache": s["v_cache"]}


def _run_mlp(s):
    ctx, lib, ok = s["ctx"].h, s["ctx"].lib, mcpm.check
    dim, f = s["x"].numel(), s["gate"].numel()
    x, gamma, xq, gate, up, hq, out = (s[n].data_ptr() for n in ("x", "gamma", "xq", "gate", "up", "hq", "out"))
    ok(lib.mcpm_rmsnorm_and_quantize_q8k(ctx, xq, x, gamma, dim, EPS))
    ok(lib.mcpm_gemv_gate_up_q4_K_q8_K(ctx, s["wg"].h, s["wu"].h, xq, gate, up, f, dim))
    ok(lib.mcpm_swiglu_and_quantize_q8k(ctx, hq, gate, up, f))
    ok(lib.mcpm_matmul_q8k(ctx, s["wd"].h, hq, f, out))
    return {"gate": s["gate"], "up": s["up"], "out": s["out"]}


def _run_head(s):
    ctx, lib, ok = s["ctx"].h, s["ctx"].lib, mcpm.check
    ok(lib.mcpm_rmsnorm(ctx, s["norm"].data_ptr(), s["x"].data_ptr(), s["gamma"].data_ptr(), s["x"].numel(), EPS))
    ok(lib.mcpm_matmul(ctx, s["w"].h, s["norm"].data_ptr(), s["logits"].data_ptr()))
    ok(lib.mcpm_argmax(ctx, s["logits"].data_ptr(), VOCAB, s["token"].data_ptr()))
    return {"norm": s["norm"], "logits": s["logits"], "token": s["token"]}


def _run_matmul(s):
    mcpm.check(s["ctx"].lib.mcpm_matmul(s["ctx"].h, s["w"].h, s["x"].data_ptr(), s["out"].data_ptr()))
    return s["out"]


def _run_sample(s):
    c = s["case"]
    mcpm.check(s["ctx"].lib.mcpm_sample_device(s["ctx"].h, s["x"].data_ptr(), c["n"], c["temperature"], c["top_p"], s["r"],
                                               s["token"].data_ptr()))
    return s["token"]


_RUN = {"greedy": _run_greedy, "first_token": _run_first_token, "turn": _run_turn, "attention": _run_attention,
        "mlp": _run_mlp, "head": _run_head, "matmul": _run_matmul, "sample": _run_sample}


def run(state):
    return _RUN[state["case"]["kind"]](state)


# ------------------------------------------------------- what a pass has to do

def _nbytes(kind, rows, cols):
    b, n = BLOCK_BYTES[kind]
    return rows * (cols // n) * b


def work(case):
    kind = case["kind"]
    if kind == "sample":
        return {"bytes": 4 * case["n"] + 4, "flops": 8 * case["n"]}
    if kind in ("attention", "mlp", "head", "matmul"):
        m = _matrices(case)
        nbytes = sum(_nbytes(*w) for w in m.values())
        flops = sum(2 * r * c for _, r, c in m.values())
        if kind == "matmul":
            nbytes += 4 * (case["rows"] + case["cols"])
        elif kind == "head":
            nbytes += 4 * (2 * MODELS[case["model"]][1] + VOCAB)
        elif kind == "mlp":
            nbytes += 4 * (3 * MODELS[case["model"]][1] + 2 * m["wg"][1])
        else:
            _, dim, nh, nkv, hd, *_ = MODELS[case["model"]]
            nbytes += 4 * (3 * dim + nh * hd + 2 * nkv * hd * case["context"])
            flops += 4 * nh * hd * case["context"]
        return {"bytes": nbytes, "flops": flops}
    L, dim, nh, nkv, hd, ffn, base, mix = MODELS[case["model"]]
    qd, kvd, f = nh * hd, nkv * hd, (ffn + 255) // 256 * 256
    # v and down are Q6_K in every layer, or, in the reference file's mix, in the layers llama.cpp gives more bits
    wide = sum(not mix or i < L // 8 or i >= 7 * L // 8 or (i - L // 8) % 3 == 2 for i in range(L))
    layer = _nbytes("q4_K", qd + kvd + 2 * ffn, dim) + _nbytes("q4_K", dim, qd)
    layer += sum(n * (_nbytes(t, kvd, dim) + _nbytes(t, dim, f)) / L for t, n in (("q6_K", wide), ("q4_K", L - wide)))
    macs = dim * (2 * qd + 2 * kvd + 2 * ffn + f)
    head = _nbytes("q6_K", VOCAB, dim)
    token = L * layer + head  # weights one token reads
    if kind == "greedy":
        tokens, pos0, prompt = case["gen"] + 1, 0, case["prompt"]
    elif kind == "turn":
        tokens, pos0, prompt = case["gen"] + 1, case["pos0"], case["new"]
    else:
        tokens, pos0, prompt = 1, 0, case["prompt"]
    end = pos0 + prompt + tokens - 1  # positions in the cache at the end
    batch = prompt - 1
    kv = 8 * kvd * L
    nbytes = (L * layer if batch else 0) + tokens * token + kv * (pos0 + batch) + kv * tokens * (end - tokens / 2) + 4 * VOCAB
    flops = 2 * L * macs * (batch + tokens) + 2 * VOCAB * dim * tokens
    flops += 4 * L * qd * (batch * (pos0 + batch / 2) + tokens * (end - tokens / 2))
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind == "sample":
        return "exact"
    if kind == "matmul":
        return {"rel": 1e-5}
    if kind in ("attention", "mlp", "head"):
        # a sum or a rotation's angle in another rounding now and then moves an activation across a rounding step
        # of its 8-bit code: 1e-3 against 64 bits at 4000 positions, 3e-7 where no code moves
        return {"rel": 4e-3, "max": 0.05}
    return {"rel": 0.02, "max": 0.2}


# --------------------------------------------------------------- in 64 bits

def _codes(x, away):
    """x through the 8-bit activation format: blocks of 256 with one scale, ties away from zero or to even."""
    v = x.view(-1, 256)
    d = v.abs().amax(dim=1, keepdim=True) / 127
    t = torch.where(d > 0, v / d, torch.zeros_like(v))
    q = torch.copysign(torch.floor(t.abs() + 0.5), t) if away else torch.round(t)
    return (q * d).view(-1)


def _rms(x, gamma):
    return x / torch.sqrt((x * x).mean() + EPS) * gamma


def _rope(x, pos, hd, base):
    i = torch.arange(0, hd, 2, device=x.device, dtype=torch.float64)
    a = pos / base ** (i / hd)
    c, s = torch.cos(a), torch.sin(a)
    p = x.view(-1, hd // 2, 2)
    return torch.stack([p[..., 0] * c - p[..., 1] * s, p[..., 0] * s + p[..., 1] * c], dim=-1).reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("attention", "mlp", "head", "matmul"):
        return None  # whole models: the activations' 8-bit codes part from any other arithmetic's within a few layers
    h, m = _inputs(case, seed), _matrices(case)

    def mul(name, x):
        t, rows, cols = m[name]
        step = max(1, (1 << 26) // cols)
        blk = cols // BLOCK_BYTES[t][1] if t != "f32" else 1
        return torch.cat([_values(t, [p[r * blk:min(rows, r + step) * blk] for p in h["parts"][name]],
                                  min(rows, r + step) - r, cols) @ x for r in range(0, rows, step)])

    x = torch.from_numpy(h["x"]).cuda().double()
    if kind == "matmul":
        return mul("w", _codes(x, False) if case["type"] in ("q4_K", "q6_K") else x)
    gamma = torch.from_numpy(h["gamma"]).cuda().double()
    if kind == "head":
        norm = _rms(x, gamma)
        logits = mul("w", _codes(norm, False))
        return {"norm": norm, "logits": logits, "token": None}
    xq = _codes(_rms(x, gamma), True)
    if kind == "mlp":
        gate, up = mul("wg", xq), mul("wu", xq)
        out = mul("wd", _codes(gate / (1 + torch.exp(-gate)) * up, True))
        return {"gate": gate, "up": up, "out": out}
    L, dim, nh, nkv, hd, ffn, base, mix = MODELS[case["model"]]
    T = case["context"]
    q, k, v = _rope(mul("wq", xq), T - 1, hd, base), _rope(mul("wk", xq), T - 1, hd, base), mul("wv", xq)
    kc, vc = (torch.from_numpy(h[n]).cuda().double() for n in ("k_cache", "v_cache"))
    kc[T - 1], vc[T - 1] = k, v
    qh = q.view(nkv, nh // nkv, hd)
    kh, vh = (c[:T].view(T, nkv, hd).permute(1, 0, 2).contiguous() for c in (kc, vc))
    p = torch.softmax(torch.bmm(qh, kh.transpose(1, 2).contiguous()) / math.sqrt(hd), dim=-1)
    att = torch.bmm(p, vh).reshape(-1)
    return {"attention": att, "out": mul("wo", _codes(att, False)), "k_cache": kc, "v_cache": vc}
