"""Batched prompt prefill on the MI355X against the oracle (marked gpu).

The reference has no prefill: its prompt loop feeds one token per call
(app/Main.hs:426-436).  So the prefill's bar is the oracle stepping the same
tokens one at a time:
- the hidden state after every layer and the logits of the last prompt
  token are within 1e-4 relative (max |a-b| / max |b|), as for a decode step;
- the next token is identical;
- the greedy ids generated after the prefill are identical to the committed
  fixtures.
The decode steps after a prefill read the K/V rows it appended, so they
check the cache contents too.
"""
from __future__ import annotations

import numpy as np
import pytest

import gemma_hip as gh
import prefill_shapes
import pyoracle as orc
from conftest import GOLDEN, rel_err

pytestmark = pytest.mark.gpu

ACT_TOL = 1e-4


def _gpu_model(ctx, cfg, seed, q4):
    m = gh.GemmaModel(ctx, cfg)
    m.synth(seed, q4)
    return m


def _oracle_model(cfg, seed, q4):
    om = orc.OracleModel(cfg)
    for name, dtype, arr in gh.synth_tensors(cfg, seed, q4):
        om.set_tensor(name, arr, dtype)
    return om


def _mini4b(mode, window=5, layers=4):
    cfg = gh.preset("gemma3-4b")
    cfg.vocab, cfg.hidden, cfg.n_layers, cfg.ffn = 2048, 512, layers, 1024
    cfg.sliding_window, cfg.global_every, cfg.max_seq, cfg.mode = window, 2, 128, mode
    return cfg


@pytest.mark.parametrize("name", ["tiny", "gemma3-1b"])
def test_prefill_matches_oracle_fixture(ctx, name):
    """Prefill of the fixture prompt: every layer of the last prompt token
    and its top-8 logits against the oracle's dump at that step; then the
    generated ids against the fixture's greedy ids."""
    fx = np.load(GOLDEN / f"{name}.npz")
    cfg = gh.preset("tiny" if name == "tiny" else "gemma3-1b")
    m = _gpu_model(ctx, cfg, int(fx["seed"]), bool(fx["q4"]))
    prompt, ids = fx["prompt"], fx["ids"]
    last = len(prompt) - 1
    dump = [int(p) for p in fx["dump_steps"]]
    assert last in dump
    i = dump.index(last)
    kv = gh.KVCache(m, 1024)
    logits, layers, nxt = gh.prefill(m, kv, prompt, want_logits=True, want_layers=True)
    assert len(kv) == len(prompt)
    for l in range(cfg.n_layers):
        err = rel_err(layers[l], fx["layers"][i][l])
        assert err < ACT_TOL, (l, err)
    assert rel_err(logits[fx["top_idx"][i]], fx["top_val"][i]) < ACT_TOL
    assert rel_err(logits[fx["topk_idx"][0]], fx["topk_val"][0]) < ACT_TOL
    assert nxt == ids[0]
    got = gh.generate(m, gh.KVCache(m, 1024), prompt, len(ids), prefill=True)
    np.testing.assert_array_equal(got, ids)


@pytest.mark.parametrize("mode", [gh.MODE_GEMMA3, gh.MODE_REF])
def test_prefill_gqa_window_then_decode_live_oracle(ctx, mode):
    """4B-shaped Q4_0 miniature (8 q heads / 4 kv heads, head_dim 256,
    window 5 that binds, global every 2nd layer): a 19-token prefill, then
    6 decode steps that attend over the prefilled K/V; every layer and the
    logits against the oracle stepping the same tokens."""
    cfg = _mini4b(mode)
    m = _gpu_model(ctx, cfg, 99, True)
    om = _oracle_model(cfg, 99, True)
    toks = gh.synth_tokens(8, "t", 25, cfg.vocab)
    n_pf = 19
    for pos in range(n_pf - 1):
        om.step(int(toks[pos]), pos)
    olog, olay, obest = om.step(int(toks[n_pf - 1]), n_pf - 1, want_layers=True)
    kv = gh.KVCache(m, 64)
    logits, layers, nxt = gh.prefill(m, kv, toks[:n_pf], want_layers=True)
    for l in range(cfg.n_layers):
        assert rel_err(layers[l], olay[l]) < ACT_TOL, l
    assert rel_err(logits, olog) < ACT_TOL
    assert nxt == obest
    for pos in range(n_pf, len(toks)):
        logits, _, layers, _ = gh.runGemmaInferenceCachedWithLayer0(m, int(toks[pos]), kv)
        olog, olay, _ = om.step(int(toks[pos]), pos, want_layers=True)
        for l in range(cfg.n_layers):
            assert rel_err(layers[l], olay[l]) < ACT_TOL, (pos, l)
        assert rel_err(logits, olog) < ACT_TOL, pos


def test_prefill_gqa_long_window_chunks_live_oracle(ctx):
    """GQA miniature (4 kv heads, group 2) with a 300-token prefill: the
    attention of each token is split over several chunks (one per 128
    positions), global layers attend to all 300 positions and local layers
    to a 160-token window; the last token's layers and logits against the
    oracle stepping the same tokens."""
    cfg = _mini4b(gh.MODE_GEMMA3, window=160, layers=2)
    cfg.max_seq = 320
    m = _gpu_model(ctx, cfg, 17, True)
    om = _oracle_model(cfg, 17, True)
    toks = gh.synth_tokens(9, "long", 300, cfg.vocab)
    for pos in range(len(toks) - 1):
        om.step(int(toks[pos]), pos)
    olog, olay, obest = om.step(int(toks[-1]), len(toks) - 1, want_layers=True)
    kv = gh.KVCache(m, 320)
    logits, layers, nxt = gh.prefill(m, kv, toks, want_layers=True)
    for l in range(cfg.n_layers):
        assert rel_err(layers[l], olay[l]) < ACT_TOL, l
    assert rel_err(logits, olog) < ACT_TOL
    assert nxt == obest


def test_prefill_passes_chunks_and_ragged_sizes(ctx):
    """f32 tiny model, 600 tokens: one prefill call (one pass), the same
    tokens as prefills of 1, 63, 65, 7 and 464 tokens, and the decode step
    token by token all reach the same last-token logits and next token; the
    caches then continue identically."""
    cfg = gh.preset("tiny")
    m = _gpu_model(ctx, cfg, 7, False)
    toks = gh.synth_tokens(11, "long", 600, cfg.vocab)
    kv_a = gh.KVCache(m, 640)
    la, _, na = gh.prefill(m, kv_a, toks)
    kv_b = gh.KVCache(m, 640)
    at = 0
    for k in (1, 63, 65, 7, 464):
        lb, _, nb = gh.prefill(m, kv_b, toks[at:at + k])
        at += k
    assert at == 600 and len(kv_a) == len(kv_b) == 600
    kv_c = gh.KVCache(m, 640)
    for t in toks:
        lc, _, nc = gh.runGemmaInferenceCached(m, int(t), kv_c)
    assert rel_err(la, lc) < ACT_TOL and rel_err(lb, lc) < ACT_TOL
    assert na == nb == nc
    ga = gh.generate(m, kv_a, [na], 6)
    gb = gh.generate(m, kv_b, [nb], 6)
    gc = gh.generate(m, kv_c, [nc], 6)
    np.testing.assert_array_equal(ga, gc)
    np.testing.assert_array_equal(gb, gc)


def test_prefill_longer_than_a_pass(ctx):
    """2100 tokens: one call (passes of 2048 + 52 rows) against the same
    tokens as prefills of 1000 and 1100, on the f32 tiny model."""
    cfg = gh.preset("tiny")
    cfg.max_seq = 2304
    m = _gpu_model(ctx, cfg, 7, False)
    toks = gh.synth_tokens(14, "pass", 2100, cfg.vocab)
    kv_a, kv_b = gh.KVCache(m, 2304), gh.KVCache(m, 2304)
    la, _, na = gh.prefill(m, kv_a, toks)
    gh.prefill(m, kv_b, toks[:1000])
    lb, _, nb = gh.prefill(m, kv_b, toks[1000:])
    assert len(kv_a) == len(kv_b) == 2100
    assert rel_err(la, lb) < ACT_TOL and na == nb


def test_prefill_longer_than_a_pass_q4(ctx):
    """The same pass boundary with Q4_0 weights and head_dim 256 (matrix-core
    attention, shared key chunks, 128-row GEMM tiles) and a 300-position
    window in the local layer: 2100 tokens as 2048 + 52 against 1000 + 1100."""
    cfg = _mini4b(gh.MODE_GEMMA3, window=300, layers=2)
    cfg.max_seq = 2304
    m = _gpu_model(ctx, cfg, 43, True)
    toks = gh.synth_tokens(17, "passq4", 2100, cfg.vocab)
    kv_a, kv_b = gh.KVCache(m, 2304), gh.KVCache(m, 2304)
    la, ya, na = gh.prefill(m, kv_a, toks, want_layers=True)
    gh.prefill(m, kv_b, toks[:1000])
    lb, yb, nb = gh.prefill(m, kv_b, toks[1000:], want_layers=True)
    for l in range(cfg.n_layers):
        assert rel_err(ya[l], yb[l]) < ACT_TOL, l
    assert rel_err(la, lb) < ACT_TOL and na == nb


@pytest.mark.parametrize("nq,nkv", [(4, 1), (8, 4)])
@pytest.mark.parametrize("n", [1010, 1900])
def test_prefill_attention_all_chunk_slots(ctx, nq, nkv, n):
    """All 16 chunk states of the matrix-core attention and its merge (1010
    tokens: 16 chunks of 64 positions; 1900: 15 of 128), in a global layer
    and in one with a 200-position window: every layer of the last token
    against the decode step fed token by token, ACT_TOL as above."""
    cfg = _mini4b(gh.MODE_GEMMA3, window=200, layers=2)
    cfg.n_heads, cfg.n_kv_heads, cfg.max_seq = nq, nkv, 1920
    m = _gpu_model(ctx, cfg, 47, True)
    toks = gh.synth_tokens(18, "slots", n, cfg.vocab)
    kv_a, kv_b = gh.KVCache(m, 1920), gh.KVCache(m, 1920)
    la, ya, na = gh.prefill(m, kv_a, toks, want_layers=True)
    for t in toks[:-1]:
        gh.runGemmaInferenceCached(m, int(t), kv_b, want_logits=False)
    lb, _, yb, nb = gh.runGemmaInferenceCachedWithLayer0(m, int(toks[-1]), kv_b)
    for l in range(cfg.n_layers):
        assert rel_err(ya[l], yb[l]) < ACT_TOL, l
    assert rel_err(la, lb) < ACT_TOL and na == nb


@pytest.mark.parametrize("nq,nkv", [(4, 4), (8, 1)])
def test_prefill_matrix_core_attention_groups_ragged_windows(ctx, nq, nkv):
    """head_dim 256 with GQA groups 1 and 8 (the 2 and 4 of the other tests
    aside): 150 tokens prefilled as pieces of 70, 1 and 79 (so later pieces
    start past position 0 and their key chunks cover earlier pieces), a
    40-token window on the local layer; the last token's logits and next
    token against the decode step fed token by token, then both caches
    continue identically."""
    cfg = _mini4b(gh.MODE_GEMMA3, window=40, layers=2)
    cfg.n_heads, cfg.n_kv_heads, cfg.max_seq = nq, nkv, 160
    m = _gpu_model(ctx, cfg, 23, True)
    toks = gh.synth_tokens(12, "fa", 150, cfg.vocab)
    kv_a = gh.KVCache(m, 160)
    at = 0
    for k in (70, 1, 79):
        la, _, na = gh.prefill(m, kv_a, toks[at:at + k])
        at += k
    kv_b = gh.KVCache(m, 160)
    for t in toks:
        lb, _, nb = gh.runGemmaInferenceCached(m, int(t), kv_b)
    assert rel_err(la, lb) < ACT_TOL and na == nb
    np.testing.assert_array_equal(gh.generate(m, kv_a, [na], 5), gh.generate(m, kv_b, [nb], 5))


@pytest.mark.parametrize("hidden,ffn,n", prefill_shapes.cases(prefill_shapes.Q4_0))
def test_prefill_gemm_tile_edges(ctx, hidden, ffn, n):
    """Q4_0 prefill GEMM in every one of its token tiles (16, 32, 64, 128
    rows) and around their edges, with one and several column splits, odd
    column block counts (hidden 288 and 1056: 9 and 33 blocks, ffn 352 and
    6944: 11 and 217) and a ragged last weight tile: the last token's layers
    and logits against the decode step fed token by token (other kernels,
    other sums; both are within ACT_TOL / 2 of the oracle elsewhere, so
    ACT_TOL bounds their difference)."""
    cfg = _mini4b(gh.MODE_GEMMA3, window=40, layers=2)
    cfg.hidden, cfg.ffn, cfg.max_seq = hidden, ffn, 400
    m = _gpu_model(ctx, cfg, 31, True)
    toks = gh.synth_tokens(13, "tile", n, cfg.vocab)
    kv_a, kv_b = gh.KVCache(m, 400), gh.KVCache(m, 400)
    la, ya, na = gh.prefill(m, kv_a, toks, want_layers=True)
    for t in toks[:-1]:
        gh.runGemmaInferenceCached(m, int(t), kv_b, want_logits=False)
    lb, _, yb, nb = gh.runGemmaInferenceCachedWithLayer0(m, int(toks[-1]), kv_b)
    for l in range(cfg.n_layers):
        assert rel_err(ya[l], yb[l]) < ACT_TOL, l
    assert rel_err(la, lb) < ACT_TOL and na == nb


@pytest.mark.parametrize("hidden,ffn,n", prefill_shapes.cases(prefill_shapes.F32))
def test_prefill_f32_gemm_tile_edges(ctx, hidden, ffn, n):
    """f32 prefill GEMM in every one of its token tiles (16, 32, 64 rows),
    below and above 512 columns, and around the edges of its rounds of column
    steps (hidden 288: 18 steps, ffn 352: 22): as the Q4_0 test above, with
    its bound."""
    cfg = _mini4b(gh.MODE_GEMMA3, window=40, layers=2)
    cfg.hidden, cfg.ffn, cfg.max_seq = hidden, ffn, 272
    m = _gpu_model(ctx, cfg, 37, False)
    toks = gh.synth_tokens(15, "f32tile", n, cfg.vocab)
    kv_a, kv_b = gh.KVCache(m, 272), gh.KVCache(m, 272)
    la, ya, na = gh.prefill(m, kv_a, toks, want_layers=True)
    for t in toks[:-1]:
        gh.runGemmaInferenceCached(m, int(t), kv_b, want_logits=False)
    lb, _, yb, nb = gh.runGemmaInferenceCachedWithLayer0(m, int(toks[-1]), kv_b)
    for l in range(cfg.n_layers):
        assert rel_err(ya[l], yb[l]) < ACT_TOL, l
    assert rel_err(la, lb) < ACT_TOL and na == nb


def _q4_rows(rows, code_blocks, scales):
    """GGUF Q4_0 bytes of `rows` equal rows: per block 32 codes and an fp16 scale."""
    d = np.asarray(scales, np.float16).reshape(-1, 1).view(np.uint8)
    q = np.asarray(code_blocks, np.uint8)
    row = np.concatenate([d, q[:, :16] | (q[:, 16:] << 4)], axis=1).reshape(-1)
    return np.tile(row, (rows, 1))


@pytest.mark.parametrize("hidden,ffn,n", [(1152, 6912, 37), (1152, 6912, 257), (1152, 6912, 1907),
                                          (2560, 10240, 1024)])
def test_prefill_q4_sums_restart(ctx, hidden, ffn, n):
    """The Q4_0 GEMM's f32 sums are restarted every 8 column blocks, so the
    down projection's error stays that of short sums.

    gate and up have equal rows, so h is one value in all ffn columns.  Even
    rows of down hold -4096 h in block 0 and 0.45 ulp of that in each other
    block; odd rows hold block 0 only.  Every product is exact.  One chain
    loses each small term that follows the large one (32 ulp over 72
    blocks).  Sums of 8 blocks, each added to a running one, round at most
    8 + nblk / 8 times, the split partials and the residual 8 + 1 times more:
    half an ulp each."""
    cfg = gh.preset("gemma3-1b")
    cfg.vocab, cfg.hidden, cfg.ffn, cfg.n_layers, cfg.max_seq = 64, hidden, ffn, 1, 2048
    cfg.flags &= ~gh.FLAG_POST_FFN_NORM
    nh, nf, one = hidden // 32, ffn // 32, np.float16(1.0)
    zero, ones = np.full((1, 32), 8), np.full((1, 32), 9)
    m = gh.GemmaModel(ctx, cfg)

    def mat(name, rows):
        m.set_tensor(name, np.ascontiguousarray(rows).reshape(-1), gh.DTYPE_Q4_0)

    def quiet(rows, nblk):
        return _q4_rows(rows, np.tile(zero, (nblk, 1)), np.full(nblk, one))

    mat("token_embd.weight", _q4_rows(64, np.tile(ones, (nh, 1)), np.full(nh, 2.0 ** -10)))
    m.set_tensor("output_norm.weight", np.ones(hidden, np.float32), gh.DTYPE_F32)
    for name, rows, nblk in (("attn_q", 1024, nh), ("attn_k", 256, nh), ("attn_v", 256, nh), ("attn_output", hidden, 32)):
        mat("blk.0.%s.weight" % name, quiet(rows, nblk))
    for name, k in (("attn_norm", hidden), ("attn_q_norm", 256), ("attn_k_norm", 256), ("post_attention_norm", hidden),
                    ("ffn_norm", hidden), ("post_ffw_norm", hidden)):
        m.set_tensor("blk.0.%s.weight" % name, np.ones(k, np.float32), gh.DTYPE_F32)
    for name in ("ffn_gate", "ffn_up"):
        mat("blk.0.%s.weight" % name, _q4_rows(ffn, np.tile(ones, (nh, 1)), np.full(nh, 0.003)))
    a = hidden * float(np.float16(0.003)) * (2.0 if cfg.flags & gh.FLAG_ZERO_CENTERED else 1.0)
    h = 0.5 * a * (1.0 + np.tanh(min(0.7978845608 * (a + 0.044715 * a ** 3), 10.0))) * a
    tiny = np.float16(0.45 * float(np.spacing(np.float32(4096.0 * h))) / h)
    codes, scales = np.full((nf, 32), 8), np.full(nf, one)
    codes[0], scales[0] = 0, np.float16(16.0)  # -8 * 32 * 16 = -4096
    odd = _q4_rows(hidden // 2, codes, scales)
    codes[1:, 5], scales[1:] = 7, tiny
    down = np.empty((hidden, nf * 18), np.uint8)
    down[0::2], down[1::2] = _q4_rows(hidden // 2, codes, scales), odd
    mat("blk.0.ffn_down.weight", down)

    _, layers, _ = gh.prefill(m, gh.KVCache(m, 2048), np.zeros(n, np.int32), want_logits=False, want_layers=True)
    out = layers[0].astype(np.float64)
    big = out[1]
    assert big < -1000.0 and np.ptp(out[0::2]) == 0.0 and np.ptp(out[1::2]) == 0.0
    ulp = float(np.spacing(np.float32(abs(big))))
    small = big * float(tiny) / 4096.0  # a block's term (the residual's share of `big` is below 1e-5)
    assert 0.43 < abs(small) / ulp < 0.47
    err = abs((out[0] - big) - (nf - 1) * small) / ulp
    assert err <= 0.5 * (8 + nf / 8 + 8 + 1), (err, small / ulp)


@pytest.mark.parametrize("ffn,n", [(128, 37), (256, 300), (480, 70)])
def test_prefill_f32_sums_restart(ctx, ffn, n):
    """Below 512 columns the f32 GEMM's sums are restarted every 16: as in the
    Q4_0 test above, down's even rows hold -4096 h in column 0 and 0.45 ulp
    of that in each other column.  A chain of 64 columns loses 28 ulp; sums
    of 16, each added to the split's running one, round at most 16 +
    columns / 16 times with the splits, the residual once or twice more."""
    cfg = gh.preset("tiny")
    cfg.vocab, cfg.ffn, cfg.n_layers = 64, ffn, 1
    cfg.flags &= ~gh.FLAG_POST_FFN_NORM
    m = gh.GemmaModel(ctx, cfg)
    H, q = cfg.hidden, cfg.n_heads * cfg.head_dim
    kv = cfg.n_kv_heads * cfg.head_dim
    down = np.zeros((H, ffn), np.float32)
    a = H * float(np.float32(0.02)) * (2.0 if cfg.flags & gh.FLAG_ZERO_CENTERED else 1.0)
    h = 0.5 * a * (1.0 + np.tanh(min(0.7978845608 * (a + 0.044715 * a ** 3), 10.0))) * a
    tiny = np.float32(0.45 * float(np.spacing(np.float32(4096.0 * h))) / h)
    down[0::2, 1:] = -tiny
    down[:, 0] = -4096.0
    for name, t in (("token_embd", np.full((64, H), 2.0 ** -10)), ("output_norm", np.ones(H)),
                    ("blk.0.attn_q", np.zeros((q, H))), ("blk.0.attn_k", np.zeros((kv, H))),
                    ("blk.0.attn_v", np.zeros((kv, H))), ("blk.0.attn_output", np.zeros((H, q))),
                    ("blk.0.ffn_gate", np.full((ffn, H), 0.02)), ("blk.0.ffn_up", np.full((ffn, H), 0.02)),
                    ("blk.0.ffn_down", down), ("blk.0.attn_norm", np.ones(H)), ("blk.0.ffn_norm", np.ones(H)),
                    ("blk.0.attn_q_norm", np.ones(cfg.head_dim)), ("blk.0.attn_k_norm", np.ones(cfg.head_dim)),
                    ("blk.0.post_attention_norm", np.ones(H)), ("blk.0.post_ffw_norm", np.ones(H))):
        m.set_tensor(name + ".weight", t.astype(np.float32).reshape(-1), gh.DTYPE_F32)
    _, layers, _ = gh.prefill(m, gh.KVCache(m, 512), np.zeros(n, np.int32), want_logits=False, want_layers=True)
    out = layers[0].astype(np.float64)
    big = out[1]
    assert big < -1000.0 and np.ptp(out[0::2]) == 0.0 and np.ptp(out[1::2]) == 0.0
    ulp = float(np.spacing(np.float32(abs(big))))
    small = big * float(tiny) / 4096.0
    assert 0.43 < abs(small) / ulp < 0.47
    err = abs((out[0] - big) - (ffn - 1) * small) / ulp
    assert err <= 0.5 * (16 + ffn / 16 + 2), (err, small / ulp)


@pytest.mark.parametrize("nq,nkv", [(4, 4), (8, 4), (4, 1), (8, 1)])
@pytest.mark.parametrize("n", [16, 97, 300])
def test_prefill_attention_chunks_outside_the_window(ctx, nq, nkv, n):
    """Chunk states of the matrix-core attention and their merge, per GQA
    group, at one chunk, at shared chunks of 16 positions and of 32 or 48
    (300 tokens: 10 or 7 chunks, most outside a 20-position window): every
    layer of the last token against the decode step, ACT_TOL as above."""
    cfg = _mini4b(gh.MODE_GEMMA3, window=20, layers=2)
    cfg.n_heads, cfg.n_kv_heads, cfg.max_seq = nq, nkv, 304
    m = _gpu_model(ctx, cfg, 41, True)
    toks = gh.synth_tokens(16, "chunk", n, cfg.vocab)
    kv_a, kv_b = gh.KVCache(m, 304), gh.KVCache(m, 304)
    la, ya, na = gh.prefill(m, kv_a, toks, want_layers=True)
    for t in toks[:-1]:
        gh.runGemmaInferenceCached(m, int(t), kv_b, want_logits=False)
    lb, _, yb, nb = gh.runGemmaInferenceCachedWithLayer0(m, int(toks[-1]), kv_b)
    for l in range(cfg.n_layers):
        assert rel_err(ya[l], yb[l]) < ACT_TOL, l
    assert rel_err(la, lb) < ACT_TOL and na == nb


def test_prefill_single_token_equals_step(ctx):
    """A prefill of one token is the decode step of that token."""
    cfg = _mini4b(gh.MODE_GEMMA3, layers=2)
    m = _gpu_model(ctx, cfg, 5, True)
    toks = gh.synth_tokens(2, "one", 3, cfg.vocab)
    kv_a, kv_b = gh.KVCache(m, 16), gh.KVCache(m, 16)
    for t in toks:
        la, _, na = gh.prefill(m, kv_a, [int(t)])
        lb, _, nb = gh.runGemmaInferenceCached(m, int(t), kv_b)
        assert rel_err(la, lb) < ACT_TOL
        assert na == nb


def test_prefill_sampling_matches_step_sampling(ctx):
    """With temperature sampling set, the prefill's next token is the draw
    the decode step makes at the same position (Philox counter = position)."""
    cfg = gh.preset("tiny")
    m = _gpu_model(ctx, cfg, 3, False)
    toks = gh.synth_tokens(4, "s", 20, cfg.vocab)
    for seed in (1, 2, 3):
        kv_a, kv_b = gh.KVCache(m, 32), gh.KVCache(m, 32)
        kv_a.set_sampling(0.8, seed)
        kv_b.set_sampling(0.8, seed)
        _, _, na = gh.prefill(m, kv_a, toks, want_logits=False)
        for t in toks:
            _, _, nb = gh.runGemmaInferenceCached(m, int(t), kv_b, want_logits=False)
        assert na == nb, seed


def test_prefill_errors_leave_cache_unchanged(ctx):
    cfg = gh.preset("tiny")
    m = _gpu_model(ctx, cfg, 1, False)
    kv = gh.KVCache(m, 8)
    gh.prefill(m, kv, [1, 2, 3])
    with pytest.raises(gh.GemmaHipError) as e:
        gh.prefill(m, kv, list(range(1, 7)))  # 3 + 6 > 8
    assert e.value.name == "GH_ERR_RANGE"
    with pytest.raises(gh.GemmaHipError) as e:
        gh.prefill(m, kv, [1, cfg.vocab])
    assert e.value.name == "GH_ERR_INVALID"
    with pytest.raises(gh.GemmaHipError) as e:
        gh.prefill(m, kv, np.zeros(0, np.int32))
    assert e.value.name == "GH_ERR_INVALID"
    with pytest.raises(gh.GemmaHipError) as e:
        gh.generate(m, kv, [1, 2, 3], 4, prefill=True)  # 3 + 3 + 3 > 8
    assert e.value.name == "GH_ERR_RANGE"
    assert len(kv) == 3
