"""GPU parity of the hybrid decode step (C ABI model) against the CPU oracle.

Bars (north star): logits within 1e-3 relative (max |dl| <= 1e-3 * max |l_ref|)
and identical greedy tokens. The fp16 KV cache is compared with the oracle's
fp16-rounded cache mode; the F32 and Q8_0 caches with the reference's own.
"""
from __future__ import annotations

import json
import os

import numpy as np
import pytest

from conftest import GOLDEN, import_into_oracle, q8_rows_close

pytestmark = pytest.mark.gpu

SMALL = dict(dim=256, hidden=768, n_layers=6, attn_layers=(1, 4), n_heads=4, n_kv=2, vocab=1024)


def rel_err(a, b):
    return float(np.max(np.abs(a.astype(np.float64) - b.astype(np.float64))) / np.max(np.abs(b)))


@pytest.fixture(scope="module")
def small_img():
    from mivi_hip.synthmodel import build_hybrid
    return build_hybrid(**SMALL, ctx_len=4096, seed=7)


def test_tiny_model_matches_reference_golden(hip, oracle):
    # tests/oracle_comparison_test.rs:14-79 on the GPU
    img = np.fromfile(os.path.join(GOLDEN, "tiny_model.gguf"), np.uint8)
    m = hip.Model(img)
    o = oracle.Model(img)
    gold = json.load(open(os.path.join(GOLDEN, "oracle_output.json")))
    for tr in gold:
        lg = m.forward(tr["token"], tr["pos"])
        lo = o.forward(tr["token"], tr["pos"])
        assert int(np.argmax(lg)) == tr["top_token"]
        assert np.all(np.abs(lg[:8] - np.array(tr["logits_sample"])) < 0.05)
        assert rel_err(lg, lo) <= 1e-3


@pytest.mark.parametrize("prec,oprec", [(0, 0), (2, 100), (1, 1)])
def test_small_model_steps_match_oracle(hip, oracle, small_img, prec, oprec):
    m = hip.Model(small_img, max_ctx=4096, kv_precision=prec)
    o = oracle.Model(small_img, max_ctx=4096, kv_precision=oprec)
    assert m.info.n_attn_layers == 2 and m.info.yarn == 0
    toks = np.random.default_rng(1).integers(0, SMALL["vocab"], 70)
    worst = 0.0
    for p, t in enumerate(toks):
        lg = m.forward(int(t), p)
        lo = o.forward(int(t), p)
        worst = max(worst, rel_err(lg, lo))
    assert worst <= 1e-3, worst


@pytest.mark.parametrize("n_heads,n_kv", [(4, 4), (12, 4)])
def test_fp16_attention_heads_per_kv_match_oracle(hip, oracle, n_heads, n_kv):
    # the fp16 matrix-core attention (P.V on v_mfma_f32_16x16x16_f16) with
    # one and three query heads per kv head (the other shapes run in the
    # tests above and the workloads: two and four), head_dim 64, 80 steps
    # over a context that crosses several 16-token groups and splits
    from mivi_hip.synthmodel import build_hybrid
    img = build_hybrid(dim=64 * n_heads, hidden=512, n_layers=3, attn_layers=(0, 2), n_heads=n_heads, n_kv=n_kv,
                       vocab=1024, ctx_len=4096, seed=31 + n_heads)
    m = hip.Model(img, max_ctx=4096, kv_precision=2)
    o = oracle.Model(img, max_ctx=4096, kv_precision=100)
    toks = np.random.default_rng(37).integers(0, 1024, 80)
    worst = 0.0
    for p, t in enumerate(toks):
        worst = max(worst, rel_err(m.forward(int(t), p), o.forward(int(t), p)))
    assert worst <= 1e-3, worst


def test_small_model_greedy_matches_oracle(hip, oracle, small_img):
    m = hip.Model(small_img, max_ctx=4096)
    o = oracle.Model(small_img, max_ctx=4096)
    prompt = np.random.default_rng(2).integers(0, SMALL["vocab"], 40)
    m.prefill(prompt[:-1])
    for p, t in enumerate(prompt[:-1]):
        o.forward_step(int(t), p, False)
    n = 64
    got = m.generate_greedy([int(prompt[-1])], [len(prompt) - 1], n)[:, 0]
    tok, want = int(prompt[-1]), []
    for i in range(n):
        lo = o.forward(tok, len(prompt) - 1 + i)
        tok = oracle.argmax(lo)
        want.append(tok)
    assert list(got) == want


def test_forward_errors(hip, small_img):
    m = hip.Model(small_img, max_ctx=128)
    with pytest.raises(hip.ModelError):
        m.forward(SMALL["vocab"], 0)          # InvalidToken (model.rs:342-344)
    with pytest.raises(hip.ModelError):
        m.forward(1, 128)                      # ContextOverflow (model.rs:345-350)


def test_batched_sequences_are_independent(hip, small_img):
    B = 4
    mb = hip.Model(small_img, max_ctx=512, max_batch=B)
    rng = np.random.default_rng(3)
    prompts = [rng.integers(0, SMALL["vocab"], 10 + 5 * b) for b in range(B)]
    for b, pr in enumerate(prompts):
        mb.prefill(pr[:-1], seq=b)
    out = mb.generate_greedy([int(p[-1]) for p in prompts], [len(p) - 1 for p in prompts], 16)
    for b, pr in enumerate(prompts):
        m1 = hip.Model(small_img, max_ctx=512)
        m1.prefill(pr[:-1])
        one = m1.generate_greedy([int(pr[-1])], [len(pr) - 1], 16)[:, 0]
        assert np.array_equal(out[:, b], one)


@pytest.mark.parametrize("B,vocab", [(3, 4096), (8, 4096), (5, 4100)])
def test_batched_full_width_matches_single_sequences(hip, B, vocab):
    # dim 2048 (the decode shapes): the packed Q6_K head (3 and 8 columns in
    # one eight-wave launch, its argmax partials per column), the multi-column Q4_K projections on the matrix cores (3 and 8
    # columns at d = 2048, 3 and 4 + 4 at d = 8192) with the RMSNorm, conv and
    # SwiGLU stages; every sequence's greedy tokens equal its own
    # single-sequence run bit for bit (a vocabulary of 4100 rows, not a
    # multiple of 32, keeps the batched head on the eight-column row quads)
    from mivi_hip.synthmodel import build_hybrid
    img = build_hybrid(dim=2048, hidden=8192, n_layers=3, attn_layers=(1,), n_heads=32, n_kv=8, vocab=vocab,
                       ctx_len=1024, seed=11)
    mb = hip.Model(img, max_ctx=256, max_batch=B)
    rng = np.random.default_rng(12)
    prompts = [rng.integers(0, vocab, 6 + 3 * b) for b in range(B)]
    for b, pr in enumerate(prompts):
        mb.prefill(pr[:-1], seq=b)
    out = mb.generate_greedy([int(p[-1]) for p in prompts], [len(p) - 1 for p in prompts], 12)
    for b, pr in enumerate(prompts):
        m1 = hip.Model(img, max_ctx=256)
        m1.prefill(pr[:-1])
        one = m1.generate_greedy([int(pr[-1])], [len(pr) - 1], 12)[:, 0]
        assert np.array_equal(out[:, b], one), (b, out[:, b], one)


@pytest.mark.parametrize("B", [3, 8])
def test_batched_column_layout_matches_gguf_rows(hip, monkeypatch, B):
    # a model with max_batch > 1 keeps its all-Q4_K projections packed in the
    # batched column kernels' group order (q|k|v, out_proj / wo, in_proj in
    # conv-channel groups, gate|up in SwiGLU groups, down); against the same
    # model on its GGUF rows (MIVI_NO_COLS_PACK) the products agree to float
    # rounding (the packed rows' min terms run on the fp16 matrix cores, and
    # the residual adds' depth slices land in any order): logits within 1e-5
    # of their largest value, same greedy tokens
    from mivi_hip.synthmodel import build_hybrid
    img = build_hybrid(dim=2048, hidden=8192, n_layers=3, attn_layers=(1,), n_heads=32, n_kv=8, vocab=4096,
                       ctx_len=1024, seed=11)
    rng = np.random.default_rng(13)
    prompts = [rng.integers(0, 4096, 5 + 2 * b) for b in range(B)]

    def run(packed):
        if packed:
            monkeypatch.delenv("MIVI_NO_COLS_PACK", raising=False)
        else:
            monkeypatch.setenv("MIVI_NO_COLS_PACK", "1")
        m = hip.Model(img, max_ctx=256, max_batch=B)
        for b, pr in enumerate(prompts):
            m.prefill(pr[:-1], seq=b)
        lg = m.forward_batch([int(p[-1]) for p in prompts], [len(p) - 1 for p in prompts])
        toks = m.generate_greedy([int(np.argmax(lg[b])) for b in range(B)], [len(p) for p in prompts], 6)
        wb = m.info.weight_bytes
        m.close()
        return lg, toks, wb

    lp, tp, wp = run(True)
    lr, tr, wr = run(False)
    assert wp > wr  # the packed copy is counted
    assert np.max(np.abs(lp - lr)) <= 1e-5 * np.max(np.abs(lr)), np.max(np.abs(lp - lr))
    assert np.array_equal(tp, tr)


@pytest.mark.parametrize("B", [2, 3, 5, 8, 11])
def test_batched_head_tiles_match_row_quads(hip, monkeypatch, B):
    # a model with max_batch > 1 keeps its Q6_K head also in 32-row tiles for
    # the batched steps (gemv_q6k_t32_kernel, v_mfma_i32_32x32x16_i8, eight
    # sequences per launch); its logits equal the row-quad heads' (which equal
    # the one-column head's) bit for bit. Q8_0 projections, whose batched
    # products are the one-column ones, keep the rest of the step
    # deterministic; 2085 tiles give some waves two tiles; 11 sequences take
    # two launches
    from mivi_hip import GgmlType
    from mivi_hip.synthmodel import build_hybrid
    vocab = 32 * 2085
    img = build_hybrid(dim=2048, hidden=2048, n_layers=2, attn_layers=(1,), n_heads=32, n_kv=8, vocab=vocab,
                       ctx_len=1024, weight_type=GgmlType.Q8_0, seed=17)
    rng = np.random.default_rng(19)
    prompts = [rng.integers(0, vocab, 4 + b) for b in range(B)]

    def run(tiles):
        if tiles:
            monkeypatch.delenv("MIVI_NO_HEAD_T32", raising=False)
        else:
            monkeypatch.setenv("MIVI_NO_HEAD_T32", "1")
        m = hip.Model(img, max_ctx=128, max_batch=B, kv_precision=2)
        for b, pr in enumerate(prompts):
            m.prefill(pr[:-1], seq=b)
        lg = m.forward_batch([int(p[-1]) for p in prompts], [len(p) - 1 for p in prompts])
        toks = m.generate_greedy([int(np.argmax(lg[b])) for b in range(B)], [len(p) for p in prompts], 4)
        wb = m.info.weight_bytes
        m.close()
        return lg, toks, wb

    lt, tt, wt = run(True)
    lq, tq, wq = run(False)
    assert wt - wq == vocab * 8 * 210  # the tile copy is counted
    assert np.array_equal(lt, lq), np.max(np.abs(lt - lq))
    assert np.array_equal(tt, tq)


@pytest.mark.parametrize("prec,oprec", [(0, 0), (2, 100), (1, 1)])
def test_chunked_prefill_matches_token_prefill_and_oracle(hip, oracle, small_img, prec, oprec):
    # PrefillStrategy::Chunked vs ::Token (model.rs:2110 tile == token): 149
    # prompt tokens in tiles of 32 (the last one ragged), then the next token's
    # logits against the token-path model and the oracle, and greedy tokens
    rng = np.random.default_rng(21)
    prompt = rng.integers(0, SMALL["vocab"], 150)
    mt = hip.Model(small_img, max_ctx=512, kv_precision=prec)
    mt.prefill(prompt[:-1])
    mc = hip.Model(small_img, max_ctx=512, kv_precision=prec)
    mc.set_prefill_strategy(32)
    mc.prefill(prompt[:-1])
    o = oracle.Model(small_img, max_ctx=512, kv_precision=oprec)
    for p, t in enumerate(prompt[:-1]):
        o.forward(int(t), p)
    n = len(prompt) - 1
    lt, lc, lo = mt.forward(int(prompt[-1]), n), mc.forward(int(prompt[-1]), n), o.forward(int(prompt[-1]), n)
    assert rel_err(lc, lt) <= 1e-3
    assert rel_err(lc, lo) <= 1e-3
    tok = int(np.argmax(lo))
    gt = mt.generate_greedy([tok], [n + 1], 8)[:, 0]
    gc = mc.generate_greedy([tok], [n + 1], 8)[:, 0]
    assert np.array_equal(gt, gc)
    # the caches and the conv state the tiles leave match the token path's
    kt, vt, ct = mt.export_state(n)
    kc, vc, cc = mc.export_state(n)
    assert np.allclose(ct, cc, rtol=1e-3, atol=1e-5)
    if prec != 1:  # float caches; Q8_0 bytes may differ where a value sits on a rounding boundary
        dt = np.float32 if prec == 0 else np.float16
        a, b = kt.view(dt).astype(np.float64), kc.view(dt).astype(np.float64)
        assert np.max(np.abs(a - b)) <= 1e-3 * np.max(np.abs(a))


def test_chunked_prefill_full_width_matrix_cores(hip):
    # dim 2048, in calls of 64 tokens (one call would be one pass of 200 rows):
    # 64 rows run the projections on the matrix cores (RMSNorm in the
    # activation split, SwiGLU and residual adds in the store), the ragged
    # last 8 the batched GEMV
    from mivi_hip.synthmodel import build_hybrid
    img = build_hybrid(dim=2048, hidden=8192, n_layers=3, attn_layers=(1,), n_heads=32, n_kv=8, vocab=4096,
                       ctx_len=1024, seed=11)
    prompt = np.random.default_rng(22).integers(0, 4096, 201)
    n = len(prompt) - 1
    mt = hip.Model(img, max_ctx=512)
    mt.prefill(prompt[:-1])
    mc = hip.Model(img, max_ctx=512)
    mc.set_prefill_strategy(64)
    for p in range(0, n, 64):
        mc.prefill(prompt[p:min(p + 64, n)], p)
    lt, lc = mt.forward(int(prompt[-1]), n), mc.forward(int(prompt[-1]), n)
    assert rel_err(lc, lt) <= 1e-3
    tok = int(np.argmax(lt))
    assert np.array_equal(mt.generate_greedy([tok], [n + 1], 8)[:, 0], mc.generate_greedy([tok], [n + 1], 8)[:, 0])


@pytest.mark.parametrize("prec,oprec", [(0, 0), (1, 1)])
def test_state_export_import_into_oracle(hip, oracle, small_img, prec, oprec):
    # cache.rs:682-914 / arena.rs:110-123 semantics: GPU-built state injected
    # into the oracle continues identically
    m = hip.Model(small_img, max_ctx=1024, kv_precision=prec)
    prompt = np.random.default_rng(4).integers(0, SMALL["vocab"], 200)
    m.prefill(prompt)
    k, v, conv = m.export_state(len(prompt))
    o = oracle.Model(small_img, max_ctx=1024, kv_precision=oprec)
    ok, ov = o.kv_views()
    row = m.kv_row_bytes()
    L = m.info.n_attn_layers
    per_layer_o = ok.size // L
    for l in range(L):
        src = slice(l * len(prompt) * row, (l + 1) * len(prompt) * row)
        ok[l * per_layer_o: l * per_layer_o + len(prompt) * row] = k[src]
        ov[l * per_layer_o: l * per_layer_o + len(prompt) * row] = v[src]
    o.conv_view()[:] = conv
    tok = int(np.random.default_rng(5).integers(0, SMALL["vocab"]))
    for i in range(8):
        lg = m.forward(tok, len(prompt) + i)
        lo = o.forward(tok, len(prompt) + i)
        assert rel_err(lg, lo) <= 1e-3
        tok = int(np.argmax(lo))
    # and back: re-import into a fresh GPU model reproduces the same logits
    m2 = hip.Model(small_img, max_ctx=1024, kv_precision=prec)
    m2.import_state(len(prompt), k, v, conv)
    m3 = hip.Model(small_img, max_ctx=1024, kv_precision=prec)
    m3.prefill(prompt)
    t0 = int(prompt[0])
    assert np.array_equal(m2.forward(t0, len(prompt)), m3.forward(t0, len(prompt)))


def test_batched_q8_kv_greedy_matches_oracle(hip, oracle, small_img):
    # config-5 semantics at small size: independent sequences, Q8_0 KV,
    # per-sequence ShortConv state; each sequence against its own oracle run
    B = 3
    m = hip.Model(small_img, max_ctx=512, kv_precision=1, max_batch=B)
    rng = np.random.default_rng(9)
    prompts = [rng.integers(0, SMALL["vocab"], 20 + 7 * b) for b in range(B)]
    for b, pr in enumerate(prompts):
        m.prefill(pr[:-1], seq=b)
    n = 24
    got = m.generate_greedy([int(p[-1]) for p in prompts], [len(p) - 1 for p in prompts], n)
    for b, pr in enumerate(prompts):
        o = oracle.Model(small_img, max_ctx=512, kv_precision=1)
        for p, t in enumerate(pr[:-1]):
            o.forward_step(int(t), p, False)
        tok, want = int(pr[-1]), []
        for i in range(n):
            lo = o.forward(tok, len(pr) - 1 + i)
            tok = oracle.argmax(lo)
            want.append(tok)
        assert list(got[:, b]) == want


def test_long_context_q8_kv_matches_oracle(hip, oracle):
    # 6000 cached tokens (many attention splits), working context 8192 (YaRN
    # active): the same synthetic Q8_0 cache and conv state in both
    from mivi_hip.synthmodel import build_hybrid
    img = build_hybrid(**SMALL, ctx_len=16384, seed=7)
    T, ctx = 6000, 8192
    m = hip.Model(img, max_ctx=ctx, kv_precision=1)
    o = oracle.Model(img, max_ctx=ctx, kv_precision=1)
    assert m.info.yarn == 1
    L, kvd = m.info.n_attn_layers, m.info.kv_dim
    k = hip.synth_random_weights(hip.GgmlType.Q8_0, 70, L * T, kvd, 1.0)
    v = hip.synth_random_weights(hip.GgmlType.Q8_0, 71, L * T, kvd, 1.0)
    conv = hip.synth_normal(72, m.conv_len(), std=0.1)
    m.import_state(T, k, v, conv)
    ok, ov = o.kv_views()
    row = m.kv_row_bytes()
    per = ok.size // L
    for l in range(L):
        ok[l * per: l * per + T * row] = k[l * T * row:(l + 1) * T * row]
        ov[l * per: l * per + T * row] = v[l * T * row:(l + 1) * T * row]
    o.conv_view()[:] = conv
    tok = 17
    for i in range(6):
        lg = m.forward(tok, T + i)
        lo = o.forward(tok, T + i)
        assert rel_err(lg, lo) <= 1e-3
        tok = int(np.argmax(lo))


def test_full_width_q8_kv_matrix_core_attention_matches_oracle(hip, oracle):
    # 32 query heads over 8 kv heads (four per kv head: every row of the int8
    # score tile in use), Q8_0 caches of 2777 and 1000 tokens (ragged 16-token
    # groups, several splits), two sequences in one batched launch; logits of
    # each sequence against its own oracle run, then batched greedy tokens
    from mivi_hip.synthmodel import build_hybrid
    img = build_hybrid(dim=2048, hidden=8192, n_layers=2, attn_layers=(1,), n_heads=32, n_kv=8, vocab=4096,
                       ctx_len=4096, seed=31)
    lens = [2777, 1000]
    m = hip.Model(img, max_ctx=4096, kv_precision=1, max_batch=2)
    L, kvd, row = m.info.n_attn_layers, m.info.kv_dim, m.kv_row_bytes()
    orc = []
    for b, T in enumerate(lens):
        k = hip.synth_random_weights(hip.GgmlType.Q8_0, 80 + 2 * b, L * T, kvd, 1.0)
        v = hip.synth_random_weights(hip.GgmlType.Q8_0, 81 + 2 * b, L * T, kvd, 1.0)
        conv = hip.synth_normal(90 + b, m.conv_len(), std=0.1)
        m.import_state(T, k, v, conv, seq=b)
        k2, v2, _ = m.export_state(T, seq=b)  # group layout on the device, the reference's rows outside
        assert np.array_equal(k2, k) and np.array_equal(v2, v)
        o = oracle.Model(img, max_ctx=4096, kv_precision=1)
        ok, ov = o.kv_views()
        per = ok.size // L
        for l in range(L):
            ok[l * per: l * per + T * row] = k[l * T * row:(l + 1) * T * row]
            ov[l * per: l * per + T * row] = v[l * T * row:(l + 1) * T * row]
        o.conv_view()[:] = conv
        orc.append(o)
    toks = [101, 2020]
    for b, T in enumerate(lens):
        lg = m.forward(toks[b], T, seq=b)
        lo = orc[b].forward(toks[b], T)
        assert rel_err(lg, lo) <= 1e-3, (b, rel_err(lg, lo))
        toks[b] = int(np.argmax(lo))
    n = 4
    got = m.generate_greedy(toks, [T + 1 for T in lens], n)
    for b, T in enumerate(lens):
        tok, want = toks[b], []
        for i in range(n):
            tok = oracle.argmax(orc[b].forward(tok, T + 1 + i))
            want.append(tok)
        assert list(got[:, b]) == want, (b, list(got[:, b]), want)


def host_sampled_loop(oracle, m, tok, pos, n_steps, cfgkw, seed, eos):
    """The generation loop of model.rs:1130-1180 on the host: the device
    decode step's logits (forward), end-of-sequence ids suppressed on the first
    token, then the oracle's Sampler::sample with the last 64 generated tokens."""
    cfg = oracle.sampler_config(**cfgkw)
    rng = oracle.Rng(seed)
    out, recent = [], []
    for s in range(n_steps):
        logits = m.forward(tok, pos + s).copy()
        if s == 0:
            logits[list(eos)] = -np.inf
        tok, _ = oracle.sample(logits, recent, cfg, rng)
        out.append(tok)
        recent = (recent + [tok])[-64:]
    return np.array(out, np.uint32)


def test_sampled_generation_matches_host_loop(hip, oracle, small_img):
    # Sampler::sample inside the captured decode step against the host loop
    # over the same device logits: the default GenerationConfig, a wider
    # nucleus with min-p and penalties, and zero temperature (greedy with
    # penalties)
    prompt = [3, 17, 250, 9, 41, 77]
    eos = (2, 5)
    # the fourth is full-vocabulary categorical sampling (top_k 0, top_p 1:
    # the split path's exp / probability kernels and the pick's categorical
    # branch, with end-of-sequence suppression, penalties from the history
    # and the next-step embedding inside the graph)
    for cfgkw, seed in ((dict(), 7), (dict(temperature=0.9, top_p=0.95, top_k=0, min_p=0.02,
                                          presence_penalty=0.3, frequency_penalty=0.2), 99),
                        (dict(temperature=0.0, repetition_penalty=1.3), 1),
                        (dict(temperature=0.9, top_p=1.0, top_k=0, min_p=0.05, repetition_penalty=1.1,
                              presence_penalty=0.3, frequency_penalty=0.2), 123)):
        m1 = hip.Model(small_img, max_ctx=128)
        m1.prefill(prompt[:-1])
        got = m1.generate([prompt[-1]], [len(prompt) - 1], 40, hip.SamplerConfig.make(**cfgkw), [seed], eos)[:, 0]
        m2 = hip.Model(small_img, max_ctx=128)
        m2.prefill(prompt[:-1])
        ref = host_sampled_loop(oracle, m2, prompt[-1], len(prompt) - 1, 40, cfgkw, seed, eos)
        assert np.array_equal(got, ref), (cfgkw, got, ref)
        assert not set(eos) & {int(got[0])}


def test_sampled_generation_greedy_config_equals_generate_greedy(hip, small_img):
    prompt = [11, 12, 13, 14]
    m1 = hip.Model(small_img, max_ctx=128)
    m1.prefill(prompt[:-1])
    g = m1.generate_greedy([prompt[-1]], [len(prompt) - 1], 32)[:, 0]
    m2 = hip.Model(small_img, max_ctx=128)
    m2.prefill(prompt[:-1])
    cfg = hip.SamplerConfig.make(temperature=0.0, repetition_penalty=1.0)
    s = m2.generate([prompt[-1]], [len(prompt) - 1], 32, cfg, [5])[:, 0]
    assert np.array_equal(g, s)


@pytest.mark.parametrize("cfgkw", [dict(temperature=0.7, top_p=0.9, top_k=50),
                                   dict(temperature=0.9, top_p=1.0, top_k=0, min_p=0.05, repetition_penalty=1.1,
                                        presence_penalty=0.3, frequency_penalty=0.2)])
def test_sampled_generation_batch_matches_single_sequences(hip, small_img, cfgkw):
    # the second configuration is full-vocabulary categorical: the batch's
    # history windows and next-step embeddings per sequence
    B = 3
    rng = np.random.default_rng(5)
    prompts = [rng.integers(0, 1024, 5 + 2 * b) for b in range(B)]
    cfg = hip.SamplerConfig.make(**cfgkw)
    mb = hip.Model(small_img, max_ctx=128, max_batch=B)
    for b, pr in enumerate(prompts):
        mb.prefill(pr[:-1], seq=b)
    out = mb.generate([int(p[-1]) for p in prompts], [len(p) - 1 for p in prompts], 24, cfg, [10 + b for b in range(B)])
    for b, pr in enumerate(prompts):
        m1 = hip.Model(small_img, max_ctx=128)
        m1.prefill(pr[:-1])
        one = m1.generate([int(pr[-1])], [len(pr) - 1], 24, cfg, [10 + b])[:, 0]
        assert np.array_equal(out[:, b], one), b


def test_full_shape_greedy_256_steps_match_oracle(hip, oracle):
    """The BASELINE decode bar at the config-4 model shape (1.2B hybrid,
    random-init Q4_K weights, Q6_K embedding/head, fp16 KV): 256 greedy
    steps from a short prompt give the oracle's tokens, and the first step's
    logits are within 1e-3 of the oracle's (relative to max |l|)."""
    from mivi_hip.synthmodel import LFM2_1B2, build_hybrid
    img = build_hybrid(**LFM2_1B2, ctx_len=65536, seed=2024)
    n, steps = 16, 256
    prompt = np.random.default_rng(21).integers(0, LFM2_1B2["vocab"], n + 1)
    m = hip.Model(img, max_ctx=n + steps + 8, kv_precision=hip.KvPrecision.F16)
    o = oracle.Model(img, max_ctx=n + steps + 8, kv_precision=oracle.KV_F16RT)
    m.prefill(prompt[:-1])
    for p, t in enumerate(prompt[:-1]):
        o.forward_step(int(t), p, False)
    lo = o.forward(int(prompt[-1]), n)
    lg = m.forward(int(prompt[-1]), n)
    assert np.max(np.abs(lg - lo)) <= 1e-3 * np.max(np.abs(lo))
    m.reset_context()
    m.prefill(prompt[:-1])
    got = m.generate_greedy([int(prompt[-1])], [n], steps)[:, 0]
    tok, want = oracle.argmax(lo), [oracle.argmax(lo)]
    for i in range(1, steps):
        tok = oracle.argmax(o.forward(tok, n + i))
        want.append(tok)
    assert list(got) == want


def oracle_from_device(oracle, img, m, n, oprec, max_ctx):
    """An oracle model holding the state the device model m built over n
    tokens (its exported caches and ShortConv state, bytes as stored)."""
    k, v, conv = m.export_state(n)
    o = oracle.Model(img, max_ctx=max_ctx, kv_precision=oprec)
    import_into_oracle(o, k, v, conv, n, m.kv_row_bytes(), m.info.n_attn_layers, f16=(oprec == 100))
    return o


@pytest.mark.parametrize("prec,oprec", [(0, 0), (2, 100), (1, 1)])
def test_qk_norm_token_and_chunked_paths_match_oracle(hip, oracle, prec, oprec):
    """transformer.rs:81-96 (token path) and :459-466 (tile path): per-head
    RMSNorm of q with attn_q_norm and of k with attn_k_norm before RoPE, as
    real LFM2 checkpoints carry them.

    F32 and fp16 caches: the logits at every prompt position on the token
    path, and the chunked path's next-token logits, against the oracle's own
    run. Q8_0 cache: a K value within rounding of a Q8_0 step quantizes to
    the neighbouring code under any other float order, and with QK-norm's
    sharp scores that moves logits by more than 1e-3 over a long prompt (the
    oracle's AVX2 and scalar kernels, both the reference's, differ by 2.6e-3
    here after 119 tokens). So the Q8_0 cache is checked code by code against
    the oracle's (each within one step, few different), and the logits
    against the oracle continuing from the device's own cache bytes. Then
    greedy tokens from the captured graph."""
    from mivi_hip.synthmodel import build_hybrid
    img = build_hybrid(**SMALL, ctx_len=4096, seed=19, qk_norm=True)
    prompt = np.random.default_rng(23).integers(0, SMALL["vocab"], 120)
    n = len(prompt) - 1
    o = oracle.Model(img, max_ctx=512, kv_precision=oprec)
    mt = hip.Model(img, max_ctx=512, kv_precision=prec)
    worst = 0.0
    for p, t in enumerate(prompt[:-1]):
        worst = max(worst, rel_err(mt.forward(int(t), p), o.forward(int(t), p)))
    # Q8_0: only a sanity bound here (the codes and the per-step arithmetic
    # are checked below)
    assert worst <= (1e-3 if prec != 1 else 1e-2), worst
    mc = hip.Model(img, max_ctx=512, kv_precision=prec)
    mc.set_prefill_strategy(32)
    mc.prefill(prompt[:-1])
    tok = int(prompt[-1])
    row, L = mt.kv_row_bytes(), mt.info.n_attn_layers
    if prec == 1:
        ko, vo = o.kv_views()
        per = ko.size // L
        for mm in (mt, mc):
            k, v, _ = mm.export_state(n)
            for l in range(L):
                assert q8_rows_close(k[l * n * row:(l + 1) * n * row], ko[l * per:l * per + n * row], n, 1, row)
                assert q8_rows_close(v[l * n * row:(l + 1) * n * row], vo[l * per:l * per + n * row], n, 1, row)
        ot, oc = oracle_from_device(oracle, img, mt, n, oprec, 512), oracle_from_device(oracle, img, mc, n, oprec, 512)
    else:
        ot = oc = o
    lo = ot.forward(tok, n)
    assert rel_err(mt.forward(tok, n), lo) <= 1e-3
    assert rel_err(mc.forward(tok, n), lo if oc is ot else oc.forward(tok, n)) <= 1e-3
    # the norm weights matter: the same model without them gives other logits
    mp = hip.Model(build_hybrid(**SMALL, ctx_len=4096, seed=19), max_ctx=512, kv_precision=prec)
    mp.prefill(prompt[:-1])
    assert rel_err(mp.forward(tok, n), lo) > 1e-2
    # 12 greedy steps from the next token (both models stand at position n + 1)
    first, want = oracle.argmax(lo), []
    t = first
    for i in range(12):
        t = oracle.argmax(ot.forward(t, n + 1 + i))
        want.append(t)
    assert list(mt.generate_greedy([first], [n + 1], 12)[:, 0]) == want
    if oc is ot:
        assert list(mc.generate_greedy([first], [n + 1], 12)[:, 0]) == want


@pytest.mark.parametrize("prec,oprec", [(2, 100), (1, 1)])
def test_qk_norm_full_width_matches_oracle(hip, oracle, prec, oprec):
    # the decode shapes (dim 2048, 32 query heads over 8 kv heads, head_dim 64)
    # with QK-norm: token path and calls of 64 tokens (the matrix-core
    # products, a ragged last call) against the oracle; the Q8_0 cache runs the matrix-core
    # attention and, as above, is checked code by code and then from the
    # device's own cache bytes
    from mivi_hip.synthmodel import build_hybrid
    img = build_hybrid(dim=2048, hidden=8192, n_layers=2, attn_layers=(1,), n_heads=32, n_kv=8, vocab=4096,
                       ctx_len=1024, seed=41, qk_norm=True)
    prompt = np.random.default_rng(24).integers(0, 4096, 151)
    n = len(prompt) - 1
    o = oracle.Model(img, max_ctx=512, kv_precision=oprec)
    for p, t in enumerate(prompt[:-1]):
        o.forward_step(int(t), p, False)
    tok = int(prompt[-1])
    ko, vo = o.kv_views()
    ko, vo = ko.copy(), vo.copy()
    lo_own = o.forward(tok, n)
    for tile in (0, 64):
        m = hip.Model(img, max_ctx=512, kv_precision=prec)
        m.set_prefill_strategy(tile)
        for p in range(0, n, tile or n):
            m.prefill(prompt[p:min(p + (tile or n), n)], p)
        if prec == 1:
            row = m.kv_row_bytes()
            k, v, _ = m.export_state(n)
            assert q8_rows_close(k, ko[:n * row], n, 1, row) and q8_rows_close(v, vo[:n * row], n, 1, row), tile
            lo = oracle_from_device(oracle, img, m, n, oprec, 512).forward(tok, n)
        else:
            lo = lo_own
        assert rel_err(m.forward(tok, n), lo) <= 1e-3, tile


@pytest.mark.parametrize("n_heads,n_kv", [(12, 3), (12, 4), (12, 6), (12, 12)])
@pytest.mark.parametrize("prec", [0, 2, 1])
def test_prefill_tile_attention_matches_per_row_attention(hip, n_heads, n_kv, prec):
    # tiles of 64 rows and more take the attention of a prefill tile (one to
    # four query heads per kv head, ragged row blocks, splits of the cached
    # tokens, later tiles over earlier ones), tiles of 32 the per-row kernels;
    # every other product of this width is the same GEMV in both, so the
    # caches and logits differ by the attention's f32 rounding alone (Q8_0
    # caches: and by values on the edge of a code, the 1e-3 bar)
    from mivi_hip.synthmodel import build_hybrid
    img = build_hybrid(dim=768, hidden=768, n_layers=4, attn_layers=(0, 2, 3), n_heads=n_heads, n_kv=n_kv, vocab=512,
                       ctx_len=2048, seed=31, qk_norm=n_kv == 4)
    prompt = np.random.default_rng(32).integers(0, 512, 1334)
    n = len(prompt) - 1
    got = []
    for tile in (32, 1100):
        m = hip.Model(img, max_ctx=2048, kv_precision=prec)
        m.set_prefill_strategy(tile)
        m.prefill(prompt[:70], 0)
        m.prefill(prompt[70:n], 70)
        k, v, conv = m.export_state(n)
        got.append((m.forward(int(prompt[-1]), n), k, v, conv))
    (la, ka, va, ca), (lb, kb, vb, cb) = got
    assert rel_err(lb, la) <= (1e-3 if prec == 1 else 2e-5)
    if prec != 1:
        dt = np.float32 if prec == 0 else np.float16
        step = 2e-5 if prec == 0 else 1e-3  # one fp16 step
        for x, y in ((ka, kb), (va, vb)):
            x, y = x.view(dt).astype(np.float64), y.view(dt).astype(np.float64)
            assert np.max(np.abs(x - y)) <= step * np.max(np.abs(x))
        assert np.max(np.abs(ca - cb)) <= 1e-4 * np.max(np.abs(ca))


@pytest.mark.parametrize("prec,oprec", [(0, 0), (2, 100), (1, 1)])
@pytest.mark.parametrize("cuts", [(70, 130, 9), (2057,), (2088,), (40, 2048, 300)])
def test_prefill_passes_full_width_match_token_path(hip, oracle, prec, oprec, cuts):
    # a model on the matrix cores at the decode shapes: prompts in several
    # calls (pos0 > 0, the ShortConv state carried, buffers that grow), one
    # pass of 2048 rows and a tail of 9 (batched GEMVs, per-row attention), of
    # 40 (matrix cores, per-row attention) and of 300 rows; K and V, the
    # ShortConv state and the next token's logits against the token path
    # (Q8_0 caches: codes within a step of the token path's, logits against
    # the oracle on the device's own cache)
    from mivi_hip.synthmodel import build_hybrid
    img = build_hybrid(dim=2048, hidden=8192, n_layers=3, attn_layers=(0, 2), n_heads=32, n_kv=8, vocab=512,
                       ctx_len=4096, seed=57)
    n = sum(cuts)
    prompt = np.random.default_rng(58).integers(0, 512, n + 1)
    mt = hip.Model(img, max_ctx=2500, kv_precision=prec)
    mt.prefill(prompt[:n])
    m = hip.Model(img, max_ctx=2500, kv_precision=prec)
    m.set_prefill_strategy(64)
    p = 0
    for c in cuts:
        m.prefill(prompt[p:p + c], p)
        p += c
    (kt, vt, ct), (k, v, conv) = mt.export_state(n), m.export_state(n)
    # float arithmetic in another order, an fp16 step (2^-10), a Q8_0 code (1 /
    # 127) of a cached value: what each may move the state by, of its largest
    tol = {0: 1e-4, 2: 2.0 ** -10, 1: 1 / 127}[prec]
    assert np.max(np.abs(ct - conv)) <= tol * np.max(np.abs(ct))
    tok, row = int(prompt[n]), m.kv_row_bytes()
    if prec == 1:
        assert q8_rows_close(k, kt, n, 2, row) and q8_rows_close(v, vt, n, 2, row)
        lo = oracle_from_device(oracle, img, m, n, oprec, 2500).forward(tok, n)
    else:
        dt = np.float32 if prec == 0 else np.float16
        for x, y in ((k, kt), (v, vt)):
            x, y = x.view(dt).astype(np.float64), y.view(dt).astype(np.float64)
            assert np.max(np.abs(x - y)) <= tol * np.max(np.abs(y))
        lo = mt.forward(tok, n)
    assert rel_err(m.forward(tok, n), lo) <= 1e-3


@pytest.mark.parametrize("t,hidden", [(1, 1000), (8, 1056), (8, 4608), (12, 4608)])
def test_prefill_swiglu_store_off_its_tiles(hip, t, hidden):
    # gate and up rows that do not fill the product's tiles of 32 pairs (F16),
    # a down projection on the GEMVs (Q8_0, 1056 columns), and the
    # loader's default widths: one pass against the token path
    from mivi_hip import GgmlType
    from mivi_hip.synthmodel import build_hybrid
    img = build_hybrid(dim=1024, hidden=hidden, n_layers=3, attn_layers=(1,), n_heads=16, n_kv=8, vocab=512, ctx_len=512,
                       seed=59, weight_type=GgmlType(t))
    prompt = np.random.default_rng(60).integers(0, 512, 131)
    n = len(prompt) - 1
    mt, m = hip.Model(img, max_ctx=512), hip.Model(img, max_ctx=512)
    mt.prefill(prompt[:n])
    m.set_prefill_strategy(64)
    m.prefill(prompt[:n])
    (kt, vt, ct), (k, v, conv) = mt.export_state(n), m.export_state(n)
    for x, y in ((k, kt), (v, vt)):
        x, y = x.view(np.float32).astype(np.float64), y.view(np.float32).astype(np.float64)
        assert np.max(np.abs(x - y)) <= 1e-4 * np.max(np.abs(y))
    assert np.max(np.abs(ct - conv)) <= 1e-4 * np.max(np.abs(ct))
    assert rel_err(m.forward(int(prompt[n]), n), mt.forward(int(prompt[n]), n)) <= 1e-4


def test_prefill_passes_keep_to_the_tile_without_matrix_cores(hip, torch_mod):
    # tiles of 64 make up passes of 2048 rows only where every projection runs
    # on the matrix cores: a model of F32 weights at their widths keeps its
    # tiles, and their buffers stay small (1500 rows: about 100 MB)
    from mivi_hip import GgmlType
    from mivi_hip.synthmodel import build_hybrid
    torch = torch_mod
    img = build_hybrid(dim=1024, hidden=4608, n_layers=2, attn_layers=(1,), n_heads=16, n_kv=8, vocab=256, ctx_len=2048,
                       seed=53, weight_type=GgmlType.F32)
    m = hip.Model(img, max_ctx=2048)
    m.set_prefill_strategy(64)
    prompt = np.random.default_rng(54).integers(0, 256, 1500)
    m.prefill(prompt[:70])
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    m.prefill(prompt)
    torch.cuda.synchronize()
    assert free - torch.cuda.mem_get_info()[0] < 16 << 20


def test_prefill_buffers_regrow_with_little_memory(hip, torch_mod):
    # a longer prompt grows the tile buffers (370 KB a row here) to twice their
    # rows; with memory left for its own rows only, it takes those, and with
    # less the call fails and the model goes on with shorter prompts
    from mivi_hip.synthmodel import build_hybrid
    torch = torch_mod
    img = build_hybrid(dim=4096, hidden=2048, n_layers=1, attn_layers=(0,), n_heads=32, n_kv=8, vocab=256, ctx_len=4096,
                       seed=55)
    prompt = np.random.default_rng(56).integers(0, 256, 4000)

    def run(m, n):
        m.reset_context()
        m.prefill(prompt[:n])
        return m.forward(int(prompt[n]), n)

    def model():
        m = hip.Model(img, max_ctx=4096)
        m.set_prefill_strategy(4096)
        return m

    m = model()
    want = run(m, 2100)
    m.close()
    m = model()
    short = run(m, 2000)
    hold = more = None
    try:
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        # 0.74 GB of buffers to come back, 0.78 needed, 1.48 for twice the rows
        hold = torch.empty(torch.cuda.mem_get_info()[0] - (400 << 20), dtype=torch.uint8, device="cuda")
        left = torch.cuda.mem_get_info()[0]
        if left > 450 << 20:  # (the allocator keeps some of its own back)
            more = torch.empty(left - (400 << 20), dtype=torch.uint8, device="cuda")
        assert torch.cuda.mem_get_info()[0] < 500 << 20
        assert np.array_equal(run(m, 2100), want)
        with pytest.raises(hip.ModelError):
            m.prefill(prompt[:3900])
        assert np.array_equal(run(m, 2000), short)
    finally:
        hold = more = None
        torch.cuda.empty_cache()
    assert np.array_equal(run(m, 2100), want)


def _patch_f32(img, name, f):
    """img with the F32 matrix `name` ([rows, cols]) changed in place by f."""
    from mivi_hip.gguf import read_tensor_index
    t, dims, off, n = read_tensor_index(img)[name]
    m = np.frombuffer(img[off:off + n].tobytes(), np.float32).reshape(dims[1], dims[0]).copy()
    f(m)
    img[off:off + n] = np.frombuffer(m.tobytes(), np.uint8)


@pytest.mark.parametrize("prec,part,big,small", [(2, "v", 3600.0, 1e-4), (0, "v", 1.6e37, 1e-36), (1, "v", 4e5, 1e-6),
                                                 (0, "k", 1.6e37, 1.0)])
def test_prefill_tile_attention_infinite_keys_and_values(hip, prec, part, big, small):
    # one prompt token whose V (K) overflows the cache's precision in one dim
    # of one kv head: the rows before it never see it (a masked token's p = 0
    # times an infinity must not reach them), the rows from it on give what the
    # per-row kernels (tiles of 32) give: infinities that end as NaN behind the
    # next norm, or, for an infinite key, scores of -inf (no weight) or +inf
    from mivi_hip import GgmlType
    from mivi_hip.synthmodel import build_hybrid
    dim, n_heads, n_kv, at, n = 768, 12, 4, 70, 100
    img = build_hybrid(dim=dim, hidden=512, n_layers=3, attn_layers=(0, 2), n_heads=n_heads, n_kv=n_kv, vocab=256,
                       ctx_len=512, seed=51, weight_type=GgmlType.F32, embd_type=GgmlType.F32)
    rng = np.random.default_rng(52)
    sign = np.where(rng.random(dim) < 0.5, -1.0, 1.0).astype(np.float32)

    def embd(m):
        m[7] = 0.02 * sign

    def proj(m):  # row 5 of kv head 1, along token 7's embedding
        m[64 + 5] = np.float32(big / np.sqrt(dim)) * sign

    def wo(m):  # the overflowing dim's share of the other tokens back to their size
        for h in range(3, 6):
            m[:, 64 * h + 5] *= np.float32(small)

    _patch_f32(img, "token_embd.weight", embd)
    _patch_f32(img, f"blk.0.attn_{part}.weight", proj)
    if part == "v":
        _patch_f32(img, "blk.0.attn_output.weight", wo)
    prompt = rng.integers(8, 256, n)
    other = prompt.copy()
    prompt[at] = 7

    def run(tokens, tile):
        m = hip.Model(img, max_ctx=512, kv_precision=prec)
        m.set_prefill_strategy(tile)
        m.prefill(tokens, 0)
        k, v, _ = m.export_state(n)
        row = m.kv_row_bytes()
        return [x.reshape(2, n, row) for x in (k, v)]

    a, ref, b = run(prompt, 128), run(prompt, 32), run(other, 128)
    dt = {0: np.float32, 2: np.float16}.get(prec)
    first = (a[1] if part == "v" else a[0])[0, at]
    if dt:
        assert np.isinf(first.view(dt)).any()
    else:
        assert np.isinf(first.reshape(-1, 34)[:, :2].copy().view(np.float16)).any()
    for x, r, y in zip(a, ref, b):
        assert np.array_equal(x[1, :64], y[1, :64])
        if dt is None:
            assert q8_rows_close(x[1, 64:at].reshape(-1), y[1, 64:at].reshape(-1), at - 64, 1, x.shape[2])
            continue
        xf, rf, yf = (z[1].copy().view(dt).astype(np.float64) for z in (x, r, y))
        tol = 2e-5 if prec == 0 else 1e-3  # f32 rounding; one fp16 step
        assert np.max(np.abs(xf[:at] - yf[:at])) <= tol * np.max(np.abs(yf[:at]))
        assert np.array_equal(np.isnan(xf[at:]), np.isnan(rf[at:]))
        fin = np.isfinite(rf[at:])
        assert np.array_equal(fin, np.isfinite(xf[at:]))
        if part == "k":
            assert fin.all()
            assert np.max(np.abs(xf[at:] - rf[at:])) <= tol * np.max(np.abs(rf[at:]))
