"""The tiled fp32-MFMA kernel: batches of more than 16 tokens over F32 caches
and over head shapes outside the MFMA kernels' (head_dim a multiple of 16 up
to 512). Each case against the oracle within the F32 (1e-3) or BF16 (5e-3)
bound: nnc's embedding call (reference model.cpp:2355-2368: the whole input
in one batch, F32, bidirectional, local layers over a symmetric window) at
EmbeddingGemma-300M's shape, causal F32 chunks over a wrapped ring, a gated
BF16 batch at head_dim 80, row blocks that end mid-token (group 3), one
split and many, and the no-alloc entry point with the partials in the fixed
scratch (bits equal to attend_device)."""
from __future__ import annotations

import numpy as np
import pytest

import libllmcpu_amd as nh
from libllmcpu_amd import hip_rt, synth

from gpu_util import errors, say

pytestmark = pytest.mark.gpu

EMB = synth.AttnConfig(5, "embeddinggemma-300m", 3, 1, 256, 24, kv_bf16=False, window=512, swa_period=6, tol=1e-3)


@pytest.mark.parametrize("layer,n", ((0, 700), (5, 700), (0, 77)))
def test_embedding_call(orc, layer, n):
    """One bidirectional batch of the whole input (local layer 0: +-256
    keys; global layer 5: every key)."""
    cfg = EMB
    window = cfg.layer_window(layer)
    K, V = synth.cache_buffer(cfg, layer, n, n)
    q = synth.qk_rows(cfg, layer, 0, np.arange(n), cfg.n_head)
    kw = dict(window=window, causal=False, n_head=cfg.n_head, n_kv=cfg.n_kv, head_dim=cfg.head_dim,
              scale=cfg.attn_scale)
    say(f"case tiled embedding layer {layer} (window {window}), {n} tokens")
    with nh.KVCache([n], [cfg.kv_dim], bf16=False) as kv:
        kv.append(0, 0, K, V)
        got = kv.attend(0, q, pos0=0, n_seq=n, **kw)
    want = orc.attend_layer(q, K, V, kv_bf16=False, rows=n, pos0=0, n_seq=n, **kw)
    ea, er = errors(got, want)
    say(f"  max-abs {ea:.3e} max-rel {er:.3e}")
    assert ea <= 1e-3


@pytest.mark.parametrize("key,layer,n_seq,pos0,n_tok", (
    ("A", 0, 3000, 2000, 1000),  # F32, head_dim 256, group 4: many splits
    ("A", 0, 200, 100, 100),  # one split
    ("C", 0, 3000, 2900, 100),  # an F32 sliding layer: a 768-row ring, wrapped
))
def test_f32_causal_chunks(orc, key, layer, n_seq, pos0, n_tok):
    base = synth.CONFIGS[key]
    cfg = synth.AttnConfig(base.index, base.name, base.n_head, base.n_kv, base.head_dim, base.n_layer, kv_bf16=False,
                           window=base.window, swa_period=base.swa_period, tol=1e-3)
    window = cfg.layer_window(layer)
    rows = cfg.layer_rows(layer, n_seq, 128)
    K, V = synth.cache_buffer(cfg, layer, rows, n_seq)
    q = synth.qk_rows(cfg, layer, 0, np.arange(pos0, pos0 + n_tok), cfg.n_head)
    kw = dict(window=window, n_head=cfg.n_head, n_kv=cfg.n_kv, head_dim=cfg.head_dim, scale=cfg.attn_scale)
    say(f"case tiled F32 {key}: rows {rows} window {window} tokens {pos0}+{n_tok}")
    with nh.KVCache([rows], [cfg.kv_dim], bf16=False) as kv:
        kv.append(0, 0, K, V)
        got = kv.attend(0, q, pos0=pos0, n_seq=pos0 + n_tok, **kw)
    want = orc.attend_layer(q, K, V, kv_bf16=False, rows=rows, pos0=pos0, n_seq=pos0 + n_tok, **kw)
    ea, er = errors(got, want)
    say(f"  max-abs {ea:.3e} max-rel {er:.3e}")
    assert ea <= 1e-3


def test_bf16_generic_shape_with_gate(orc):
    """head_dim 80, 24 query heads over 8 KV heads (group 3: a 64-row block
    ends mid-token), 300 tokens, Qwen3.5's output gate."""
    cfg = synth.AttnConfig(12, "hd80 g3", 24, 8, 80, 1)
    n_seq, pos0, n_tok = 1500, 1200, 300
    K, V = synth.cache_buffer(cfg, 0, n_seq, n_seq)
    q = synth.qk_rows(cfg, 0, 0, np.arange(pos0, pos0 + n_tok), cfg.n_head)
    gate = np.random.default_rng(5).standard_normal(q.shape).astype(np.float32)
    kw = dict(n_head=cfg.n_head, n_kv=cfg.n_kv, head_dim=80, scale=cfg.attn_scale)
    say("case tiled BF16 head_dim 80, group 3, gated, 300 tokens")
    with nh.KVCache([n_seq], [cfg.kv_dim]) as kv:
        kv.append(0, 0, K, V)
        got = kv.attend(0, q, pos0=pos0, n_seq=pos0 + n_tok, gate=gate, **kw)
    want = orc.attend_layer(q, K, V, kv_bf16=True, rows=n_seq, pos0=pos0, n_seq=pos0 + n_tok, **kw)
    want = want / (1.0 + np.exp(-gate.astype(np.float64)))
    ea, er = errors(got, want)
    say(f"  max-abs {ea:.3e}")
    assert ea <= 5e-3


def test_tiled_noalloc_matches_attend_device(orc):
    """A 200-token F32 batch through nnc_hip_attend_device_noalloc (partials
    in the library's fixed array) gives attend_device's bits."""
    cfg = synth.CONFIGS["A"]
    n_seq, pos0, n_tok = 1024, 824, 200
    K, V = synth.cache_buffer(cfg, 0, n_seq, n_seq)
    q = synth.qk_rows(cfg, 0, 0, np.arange(pos0, pos0 + n_tok), cfg.n_head)
    kw = dict(n_head=cfg.n_head, n_kv=cfg.n_kv, head_dim=cfg.head_dim, scale=cfg.attn_scale)
    with nh.KVCache([n_seq], [cfg.kv_dim], bf16=False) as kv:
        kv.append(0, 0, K, V)
        q_dev, o_a, o_b = hip_rt.malloc(q.nbytes), hip_rt.malloc(q.nbytes), hip_rt.malloc(q.nbytes)
        try:
            hip_rt.to_device(q_dev, q)
            say("case tiled F32 200 tokens: attend_device and the no-alloc form")
            kv.attend_device(0, q_dev, o_a, n_tok=n_tok, pos0=pos0, **kw)
            kv.attend_device_noalloc(0, q_dev, o_b, n_tok=n_tok, pos0=pos0, **kw)
            kv.sync()
            a = hip_rt.to_host(np.empty_like(q), o_a)
            b = hip_rt.to_host(np.empty_like(q), o_b)
        finally:
            for d in (q_dev, o_a, o_b):
                hip_rt.free(d)
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    want = orc.attend_layer(q, K, V, kv_bf16=False, rows=n_seq, pos0=pos0, n_seq=pos0 + n_tok, **kw)
    assert errors(a, want)[0] <= 1e-3


# Both sides of the rule for the three-part bf16 products (512 rows per KV head,
# 4000 in all and enough keys; 128-row blocks, 32-key groups): the smallest
# batch that takes them and one token less, ragged last blocks, one split and
# many, windows on both sides, rings that have wrapped, spans that start
# mid-group.
T3_CASES = (
    # n_head, n_kv, head_dim, causal, window, n_seq, n_tok, ring
    (4, 1, 256, True, 0, 1011, 1000, False),
    (4, 1, 256, True, 0, 1010, 999, False),
    (3, 1, 256, False, 512, 1400, 1400, False),
    (3, 1, 256, False, 0, 1337, 1337, False),
    (16, 8, 128, True, 0, 1333, 261, False),
    (16, 8, 128, True, 300, 1500, 300, True),
    (8, 2, 64, True, 0, 555, 501, False),
    (32, 8, 64, False, 200, 150, 150, False),
    (4, 4, 256, True, 700, 2600, 1003, True),
    # (the cases above of little work, or whose operands leave no room for
    # splits, run the fp32 products; these the three-part ones)
    (4, 1, 256, True, 700, 2600, 1003, True),
    (16, 8, 128, True, 300, 1500, 900, True),
    (8, 2, 64, True, 600, 2600, 1003, True),
    (8, 2, 64, True, 0, 1055, 1001, False),
    (32, 8, 64, False, 400, 600, 600, False),
)


@pytest.mark.parametrize("c", T3_CASES, ids=lambda c: "-".join(map(str, c)))
def test_f32_three_part_products(orc, c):
    """Against the oracle to 2e-5: fp32 products and sums on both sides (the
    scores' fp32 rounding at |s| up to ~30 log2 units, about 30 * 2^-23 = 4e-6
    per weight, on outputs up to ~4); the no-alloc entry point runs the same
    launches, bit for bit; a gate on top."""
    n_head, n_kv, hd, causal, window, n_seq, n_tok, ring = c
    cfg = synth.AttnConfig(61, "t3", n_head, n_kv, hd, 1, kv_bf16=False, window=window, swa_period=2, tol=1e-3)
    rows = nh.kv_rows(4 * n_seq, window, n_tok) if ring else n_seq + 5
    pos0 = n_seq - n_tok
    K, V = synth.cache_buffer(cfg, 0, rows, n_seq)
    q = synth.qk_rows(cfg, 0, 0, np.arange(pos0, n_seq), n_head)
    kw = dict(window=window, causal=causal, n_head=n_head, n_kv=n_kv, head_dim=hd, scale=cfg.attn_scale)
    say(f"case three-part {c}: rows {rows}")
    gate = np.random.default_rng(1).standard_normal(q.shape).astype(np.float32)
    with nh.KVCache([rows], [cfg.kv_dim], bf16=False) as kv:
        kv.append(0, 0, K, V)
        got = kv.attend(0, q, pos0=pos0, n_seq=n_seq, **kw)
        gated = kv.attend(0, q, pos0=pos0, n_seq=n_seq, gate=gate, **kw)
        qd, od = hip_rt.malloc(q.nbytes), hip_rt.malloc(q.nbytes)
        try:
            hip_rt.to_device(qd, q)
            kv.attend_device_noalloc(0, qd, od, n_tok=n_tok, pos0=pos0, n_seq=n_seq, **kw)
            kv.sync()
            fixed = hip_rt.to_host(np.empty_like(got), od)
        finally:
            hip_rt.free(qd)
            hip_rt.free(od)
    want = orc.attend_layer(q, K, V, kv_bf16=False, rows=rows, pos0=pos0, n_seq=n_seq, **kw)
    ea, er = errors(got, want)
    say(f"  max-abs {ea:.3e} max-rel {er:.3e}")
    assert ea <= 2e-5
    assert np.array_equal(fixed.view(np.uint32), got.view(np.uint32))
    assert np.abs(gated - got / (1 + np.exp(-gate.astype(np.float64)))).max() <= 2e-6


def test_f32_three_part_products_in_a_graph(orc):
    """Captured before its scratch has grown a long F32 batch with one split
    runs the fp32 kernel; replays agree with each other and, to 2e-5, with the
    eager call."""
    n_head, n_kv, hd, n = 64, 16, 64, 700  # (176 row blocks of 64 and 16 KV heads: one split)
    cfg = synth.AttnConfig(62, "t3 graph", n_head, n_kv, hd, 1, kv_bf16=False)
    K, V = synth.cache_buffer(cfg, 0, n, n)
    q = synth.qk_rows(cfg, 0, 0, np.arange(n), n_head)
    kw = dict(n_tok=n, pos0=0, n_head=n_head, n_kv=n_kv, head_dim=hd, scale=cfg.attn_scale)
    with nh.KVCache([n], [cfg.kv_dim], bf16=False) as kv:
        kv.append(0, 0, K, V)
        qd, od = hip_rt.malloc(q.nbytes), hip_rt.malloc(q.nbytes)
        try:
            hip_rt.to_device(qd, q)
            say("case three-part under capture")
            g = hip_rt.Graph(kv.stream, lambda: kv.attend_device(0, qd, od, **kw))
            first = None
            for _ in range(3):
                hip_rt.to_device(od, np.zeros_like(q))
                g.launch(kv.stream)
                kv.sync()
                got = hip_rt.to_host(np.empty_like(q), od)
                first = got if first is None else first
                assert np.array_equal(got, first)
            g.close()
            kv.attend_device(0, qd, od, **kw)
            kv.sync()
            assert np.abs(hip_rt.to_host(np.empty_like(q), od) - first).max() <= 2e-5
        finally:
            hip_rt.free(qd)
            hip_rt.free(od)


def test_f32_three_part_special_values():
    """Infinities, NaN and large values in K and V, every key attended: the same classes (finite, +inf, -inf, NaN) per element as shorter
    batches of the same tokens, which run fp32 products, and the finite ones
    within 2e-5 of theirs."""
    n_head, n_kv, hd, n = 4, 1, 256, 1024
    cfg = synth.AttnConfig(63, "t3 special", n_head, n_kv, hd, 1, kv_bf16=False)
    K, V = synth.cache_buffer(cfg, 0, n, n)
    K, V = K.copy(), V.copy()
    V[17, 3], V[400, 4], V[900, 5] = np.inf, -np.inf, np.nan
    # (a weight reaches 2^8 against its row's offset, and up to 1024 of them are
    # summed before the division: both kernels are finite up to the limit / 2^18)
    V[33, 6], V[33, 7] = np.finfo(np.float32).max / 2**18, -np.finfo(np.float32).max / 2**18
    q = synth.qk_rows(cfg, 0, 0, np.arange(n), n_head)
    q.reshape(n, n_head, hd)[:, :, 9] = np.abs(q.reshape(n, n_head, hd)[:, :, 9]) + 0.1
    K[55, 9] = -np.inf  # (weight 0 in every row)
    kw = dict(n_seq=n, causal=False, n_head=n_head, n_kv=n_kv, head_dim=hd, scale=cfg.attn_scale)
    say("case three-part special values")
    with nh.KVCache([n], [cfg.kv_dim], bf16=False) as kv:
        kv.append(0, 0, K, V)
        got = kv.attend(0, q, pos0=0, **kw)
        want = np.concatenate([kv.attend(0, q[i:i + 256], pos0=i, **kw) for i in range(0, n, 256)])
    for cls in (np.isfinite, np.isposinf, np.isneginf, np.isnan):
        say(f"  {cls.__name__}: columns that differ {np.unique(np.argwhere(cls(got) != cls(want))[:, 1] % hd)}")
        assert np.array_equal(cls(got), cls(want)), cls.__name__
    assert np.isposinf(want).any() and np.isnan(want).any()
    ok = np.isfinite(want)
    g, w = got[ok].astype(np.float64), want[ok].astype(np.float64)
    assert (np.abs(g - w) <= 2e-5 * (1 + np.abs(w))).all()


@pytest.mark.parametrize("c", ((4, 1, 256, True, 0), (4, 1, 256, True, 420), (16, 8, 128, True, 0), (16, 8, 128, False, 400),
                               (8, 8, 64, True, 0), (16, 8, 64, False, 401)), ids=lambda c: "-".join(map(str, c)))
def test_f32_three_part_non_finite_v_stays_with_its_rows(c):
    """An infinite or NaN V row changes no token that does not attend it (to 2e-5:
    the rows of a work-group that has such a key run in fp32), whichever block,
    key group or split the key shares with it; those that attend it are not finite."""
    n_head, n_kv, hd, causal, window = c
    n = 1100
    cfg = synth.AttnConfig(65, "t3 reach", n_head, n_kv, hd, 1, kv_bf16=False, window=window, swa_period=2)
    K, V = synth.cache_buffer(cfg, 0, n, n)
    q = synth.qk_rows(cfg, 0, 0, np.arange(n), n_head)
    kw = dict(pos0=0, n_seq=n, window=window, causal=causal, n_head=n_head, n_kv=n_kv, head_dim=hd, scale=cfg.attn_scale)
    span = [nh.attn_span(causal, window, t, n) for t in range(n)]
    with nh.KVCache([n], [cfg.kv_dim], bf16=False) as kv:
        say(f"case three-part reach of non-finite V {c}")
        kv.append(0, 0, K, V)
        want = kv.attend(0, q, **kw)
        for k, x in ((333, np.inf), (511, np.nan), (640, -np.inf), (1003, np.nan)):
            kv.append(0, k, K[k:k + 1], np.full_like(V[k:k + 1], x))
            got = kv.attend(0, q, **kw)
            kv.append(0, k, K[k:k + 1], V[k:k + 1])
            dirty = np.array([lo <= k <= hi for lo, hi in span])
            same = (np.abs(got - want) <= 2e-5 * (1 + np.abs(want))).all(1)
            say(f"  key {k}: attended by {dirty.sum()} tokens; others changed {np.flatnonzero(~dirty & ~same)[:40]}")
            assert (~dirty).sum() > 50 and same[~dirty].all()
            assert not np.isfinite(got[dirty]).any()


def test_f32_three_part_infinite_scores():
    """Infinite K against large Q elements, and infinite Q against large K ones, of
    either sign in their second bf16 part: scores of -inf weigh 0 and rows whose
    every score is -inf are 0, as in shorter batches, which run fp32 products."""
    n_head, n_kv, hd, n = 4, 1, 256, 1024
    cfg = synth.AttnConfig(66, "t3 infinite scores", n_head, n_kv, hd, 1, kv_bf16=False)
    K, V = synth.cache_buffer(cfg, 0, n, n)
    q = synth.qk_rows(cfg, 0, 0, np.arange(n), n_head)
    rng = np.random.default_rng(4)
    large = (rng.uniform(4e3, 9e4, (n, n_head))).astype(np.float32)
    kw = dict(n_seq=n, causal=False, n_head=n_head, n_kv=n_kv, head_dim=hd, scale=cfg.attn_scale)
    for what in ("K", "Q"):
        k1, q1 = K.copy(), q.copy()
        if what == "K":
            k1[:, 9], k1[55, 9] = 0, -np.inf
            q1.reshape(n, n_head, hd)[:, :, 9] = large
        else:
            k1[:, 9] = -large[:, 0] / 512  # (below 2^8)
            q1.reshape(n, n_head, hd)[:, :, 9] = 0
            q1.reshape(n, n_head, hd)[::7, :, 9] = np.inf
        say(f"case three-part infinite {what}")
        with nh.KVCache([n], [cfg.kv_dim], bf16=False) as kv:
            kv.append(0, 0, k1, V)
            got = kv.attend(0, q1, pos0=0, **kw)
            want = np.concatenate([kv.attend(0, q1[i:i + 256], pos0=i, **kw) for i in range(0, n, 256)])
        assert np.isfinite(want).all()
        assert (np.abs(got - want) <= 2e-5 * (1 + np.abs(want))).all(), what
        assert what == "K" or (want[::7] == 0).all()
