"""Batched prompt processing (mcpm_engine_prefill, MFMA GEMMs) against the
per-token decode path: the KV cache rows of every layer must be bit-identical
to those left by one forward per token, and the generated continuation the
same.  The per-token path itself is checked against the oracle elsewhere;
the greedy test below also checks prefill + decode against the oracle."""
import os
import subprocess

import numpy as np
import pytest

import mcpm
import oracle as O
from conftest import ROOT, announce, assert_bits

pytestmark = pytest.mark.gpu

# (layers, dim, heads, kv heads, head_dim, ffn, vocab, mix, prompt length)
CASES = [
    (2, 2304, 32, 8, 64, 5760, 4096, 0, 100),   # 2.4B layer shape, Q6_K v/down, crosses a 64-position chunk
    (3, 2304, 32, 8, 64, 5760, 4096, 1, 40),    # llama-style mix: Q4_K down in some layers
    (2, 512, 8, 2, 64, 1400, 2000, 0, 300),     # q-dim 512 (2 blocks), 5 attention chunks
    (2, 256, 4, 2, 64, 512, 300, 0, 130),       # q-dim 256 (1 block), ffn padded 512
    (2, 512, 8, 2, 64, 1400, 2000, 0, 1100),    # two batched passes (1024 + 75 tokens), 18 chunks
]


def _run(eng, prompt, n_gen, prefill):
    eng.set_prefill(prefill)
    eng.init_kv_cache(len(prompt) + n_gen + 4)
    toks = list(eng.generate_greedy(prompt, n_gen))
    kv = [eng.read_kv(l, 0, len(prompt) - 1) for l in range(eng.cfg.n_layers)]
    return toks, kv


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"L{c[0]}-d{c[1]}-h{c[2]}-mix{c[7]}-p{c[8]}")
def test_prefill_kv_and_tokens_match_per_token(ctx, case):
    L, D, NH, NKV, HD, F, V, mix, n_prompt = case
    cfg = mcpm.make_config(L, D, NH, NKV, HD, F, V)
    img = mcpm.synth_gguf(cfg, seed=4242, mix=mix)
    prompt = np.random.default_rng(7).integers(0, V, n_prompt).astype(np.int32)
    announce(f"prefill case {case}")
    eng = mcpm.Engine(ctx, image=img)
    try:
        want_toks, want_kv = _run(eng, prompt, 6, prefill=False)
        got_toks, got_kv = _run(eng, prompt, 6, prefill=True)
    finally:
        eng.free()
    for l in range(L):
        assert_bits(got_kv[l][0], want_kv[l][0])
        assert_bits(got_kv[l][1], want_kv[l][1])
    assert got_toks == want_toks


# Prompt lengths around the GEMM's 16-token tiles and their grouping (one to
# four tiles per work group, a last group that is not full) at shapes whose rows
# end inside a row tile or pair (ffn 1400 and 520; 1401 and 7, whose activations
# also start at 4-byte offsets), and rows enough for row tiles in pairs (2304 at
# 200 tokens and more).
TILE_CASES = [(2, 512, 8, 2, 64, 1400, 2000, mix, n) for mix in (0, 1) for n in (2, 16, 17, 18, 33, 34, 50, 65, 66, 82, 114)]
TILE_CASES += [(2, 256, 4, 1, 64, 520, 300, 0, 37), (2, 256, 4, 1, 64, 1401, 300, 0, 21), (2, 256, 4, 1, 64, 7, 300, 0, 19), (2, 2304, 32, 8, 64, 5760, 1000, 0, 241), (2, 2304, 32, 8, 64, 5760, 1000, 1, 337)]


@pytest.mark.parametrize("case", TILE_CASES, ids=lambda c: f"d{c[1]}-hd{c[4]}-mix{c[7]}-p{c[8]}")
def test_prefill_token_tiles(ctx, case):
    test_prefill_kv_and_tokens_match_per_token(ctx, case)


# Row tiles in pairs at one, two and three token tiles, which take 8192 rows: o and
# down (Q4_K, Q6_K; rows of 32 blocks, past the quantization's 24) and q, k and v
WIDE_CASES = [(2, 8192, 4, 1, 64, 256, 300, 0, n) for n in (10, 26, 42)] + [(2, 256, 128, 16, 64, 256, 300, 0, n) for n in (10, 26)]


@pytest.mark.parametrize("case", WIDE_CASES, ids=lambda c: f"d{c[1]}-h{c[2]}-p{c[8]}")
def test_prefill_wide_matrices(ctx, case):
    test_prefill_kv_and_tokens_match_per_token(ctx, case)


# head_dim 128 and 96 (the attention's instances past 64), 32 (below), groups of 8, 3 and 1 query heads,
# contexts that end inside a chunk, at its edge and one past it
ATTN_CASES = [(2, 512, 16, 2, 128, 512, 300, 0, 70), (2, 512, 8, 4, 96, 512, 300, 0, 66), (2, 512, 8, 1, 32, 512, 300, 0, 65),
              (2, 768, 12, 4, 64, 512, 300, 0, 130), (2, 256, 4, 4, 64, 512, 300, 0, 64), (2, 512, 16, 2, 128, 512, 300, 0, 333)]
# groups that do not divide a wave's 16 rows: 5, 6 and 7 query heads, a last token tile that is not full
ATTN_CASES += [(2, 512, 20, 4, 64, 512, 300, 0, 90), (2, 512, 24, 4, 64, 512, 300, 0, 131), (2, 512, 28, 4, 64, 512, 300, 0, 77)]


@pytest.mark.parametrize("case", ATTN_CASES, ids=lambda c: f"h{c[2]}-kv{c[3]}-hd{c[4]}-p{c[8]}")
def test_prefill_attention_shapes(ctx, case):
    test_prefill_kv_and_tokens_match_per_token(ctx, case)


# normal, widely spread, softmax terms down to denormals, products that underflow, denormal values, sums that cancel
@pytest.mark.parametrize("distribution", range(6))
def test_fp32_mfma_is_the_fma_chain(distribution):
    announce(f"fp32 mfma distribution {distribution}")
    r = subprocess.run([os.path.join(ROOT, "tests", "cpp", "mfma_check"), str(distribution)], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert ", 0 differ" in r.stdout


def test_prefill_infinite_v_leaves_earlier_tokens(ctx):
    """A V row with infinities weighs 0 in the tokens before it: they keep their bits (0 * inf would be NaN)."""
    cfg = mcpm.make_config(2, 512, 8, 2, 64, 512, 300)
    img = mcpm.synth_gguf(cfg, seed=11, mix=0).copy()
    _, T = O.read_gguf(img)
    # dimension 0 of the embedding is 0 but for token 299, and layer 0's norm
    # scales it by 1e38, so that only that token's V overflows; q is 0, so
    # every score is 0 and the token's K takes no part
    embd = T["token_embd.weight"][2].reshape(300, 2, 210)
    embd[:, 0, 0] &= 0xF0
    embd[:, 0, 128] = (embd[:, 0, 128] & 0xFC) | 2
    embd[299, 0, 0] |= 0x0F
    embd[299, 0, 128] |= 3
    T["blk.0.attn_norm.weight"][2].view(np.float32)[0] = 1e38
    T["blk.0.attn_q.weight"][2].reshape(-1, 144)[:, :4] = 0
    T["blk.0.attn_v.weight"][2].reshape(-1, 210)[:, 208:] = np.array([0x2E66], np.uint16).view(np.uint8)  # d = 0.1
    prompt = np.random.default_rng(5).integers(0, 299, 60).astype(np.int32)
    prompt[37] = 299
    eng = mcpm.Engine(ctx, image=img)
    try:
        kv = {}
        for prefill in (False, True):
            eng.set_prefill(prefill)
            eng.init_kv_cache(64)
            eng.generate_greedy(prompt, 1)
            kv[prefill] = [eng.read_kv(l, 0, 59) for l in range(2)]
    finally:
        eng.free()
    v0 = kv[False][0][1].reshape(59, -1)
    assert not np.isfinite(v0[37]).all() and np.isfinite(np.delete(v0, 37, axis=0)).all()
    assert_bits(kv[True][0][1], kv[False][0][1])
    for i in range(2):
        assert np.isfinite(kv[False][1][i][:37]).all()
        assert_bits(kv[True][1][i][:37], kv[False][1][i][:37])


def test_prefill_greedy_matches_oracle(ctx):
    cfg = mcpm.make_config(2, 512, 8, 2, 64, 1400, 2000)
    img = mcpm.synth_gguf(cfg, seed=31, mix=0)
    prompt = [int(t) for t in np.random.default_rng(3).integers(0, 2000, 70)]
    announce("prefill greedy vs oracle")
    eng = mcpm.Engine(ctx, image=img)
    try:
        eng.set_prefill(True)
        eng.init_kv_cache(96)
        got = list(eng.generate_greedy(prompt, 10))
    finally:
        eng.free()
    om = O.OracleModel(img)
    want = list(om.generate_greedy(prompt, 10))
    om.close()
    assert got == want


def test_prefill_sampled_matches_per_token(ctx):
    cfg = mcpm.make_config(2, 512, 8, 2, 64, 1400, 2000)
    img = mcpm.synth_gguf(cfg, seed=5, mix=0)
    prompt = np.random.default_rng(11).integers(0, 2000, 90).astype(np.int32)
    announce("prefill sampled")
    eng = mcpm.Engine(ctx, image=img)
    try:
        out = []
        for pf in (False, True):
            eng.set_prefill(pf)
            eng.init_kv_cache(128)
            out.append(list(eng.generate_sampled(prompt, 16, 0.8, 0.95, 1234)))
    finally:
        eng.free()
    assert out[0] == out[1]


def test_prefill_rejects_bad_arguments(ctx):
    cfg = mcpm.make_config(1, 256, 4, 2, 64, 512, 300)
    eng = mcpm.Engine(ctx, image=mcpm.synth_gguf(cfg, seed=1))
    try:
        with pytest.raises(mcpm.McpmError):
            eng.prefill([1, 2, 3])  # no KV cache yet
        eng.init_kv_cache(8)
        with pytest.raises(mcpm.McpmError):
            eng.prefill(list(range(9)))  # past the capacity
        with pytest.raises(mcpm.McpmError):
            eng.prefill([0, 300])  # token out of range
        eng.prefill([])
    finally:
        eng.free()
