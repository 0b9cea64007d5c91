"""Timed cases of the framework's main paths, through its public entry points.

A case is one of four kinds of work that an inference program gives this
library, over the range of sizes such programs use:

- "attend": the attention calls of a pass over `layers` layers whose K/V are
  already in the cache: decode (one token), a session batch (2 to 16 tokens),
  prefill chunks, a whole bidirectional input (the embedding call);
- "layer": the whole attention half of a layer: q, k and v projections, the
  pre-attention step (norms, RoPE, append), attention, output projection;
- "proj": a layer's weight products (q/k/v, o, gate/up, down);
- "head": the vocabulary projection: the logits of a batch, or for one vector
  the logits and the greedy token.

Head shapes are those of the models this repository's benchmark and tests
name. Weights, activations and cached rows are random with the scales the
models have: per-head normalised q and k, unit-variance v and activations.
"""
import math

import numpy as np
import torch

from libllmcpu_amd import KVCache, NncHipPrep, kv_rows, load_library

DEV = "cuda"

# (n_head, n_kv, head_dim) of the models the benchmark names, with the width of
# the residual stream and of the MLP where projections are timed.
LLAMA = dict(n_head=32, n_kv=8, head_dim=64)
QWEN = dict(n_head=32, n_kv=8, head_dim=128)
GEMMA_1B = dict(n_head=4, n_kv=1, head_dim=256)
GEMMA_4B = dict(n_head=8, n_kv=4, head_dim=256)
EMBED = dict(n_head=3, n_kv=1, head_dim=256)


def _attend(name, shape, *, layers, pos0, chunk, chunks=1, bf16=True, window=0, period=0, causal=True):
    c = dict(kind="attend", layers=layers, pos0=pos0, chunk=chunk, chunks=chunks, bf16=bf16, window=window,
             period=period, causal=causal, **shape)
    return dict(c, name=name) if name else c


def listed():
    return [
        # Gemma-3-270M's decode step over an F32 cache: the shortest calls, bound by latency and launches.
        _attend("decode_f32_1k", GEMMA_1B, layers=18, pos0=1023, chunk=1, bf16=False),
        # Qwen3-4B's decode step at long context: K and V streamed from HBM.
        _attend("decode_qwen_32k", QWEN, layers=12, pos0=32767, chunk=1),
        # A 16-token forward pass of a session (verification of drafts, or a short prompt) far into a context.
        _attend("session_qwen_20k", QWEN, layers=12, pos0=20011, chunk=16),
        # A 4096-token prompt in 512-token chunks.
        _attend("prefill_qwen_4k", QWEN, layers=2, pos0=0, chunk=512, chunks=8),
        # The last 1024-token chunk of a 16k prompt on five sliding layers and a global one.
        _attend("prefill_gemma_16k", GEMMA_4B, layers=6, pos0=15360, chunk=1024, window=1024, period=6),
        # A ragged chunk after a short history, head_dim 64.
        _attend("prefill_llama_ragged", LLAMA, layers=16, pos0=733, chunk=317),
        # An embedding call: a whole 2048-token input, bidirectional, F32 K/V, five of six layers windowed.
        _attend("embed_f32_2k", EMBED, layers=6, pos0=0, chunk=2048, bf16=False, window=512, period=6, causal=False),
        # The attention half of Llama-3.2-1B's decode step: small products and short attention, launch by launch.
        dict(name="layer_decode_llama", kind="layer", layers=16, pos0=4000, n_tok=1, fmt="bf16", n_embd=2048, **LLAMA),
        # The attention half of two Qwen3-4B layers on a prompt chunk: large products beside prefill attention.
        dict(name="layer_prefill_qwen", kind="layer", layers=2, pos0=1536, n_tok=512, fmt="bf16", n_embd=2560, **QWEN),
        # Qwen3-4B's weight products in the 4-bit layout, one vector (decode).
        dict(name="proj_q4s_decode", kind="proj", layers=6, fmt="q4_s", n_vec=1, n_embd=2560, q_dim=4096, kv_dim=1024,
             n_ff=9728),
        # The same in the 8-bit layout for a session batch.
        dict(name="proj_q8_session", kind="proj", layers=4, fmt="q8_0", n_vec=16, n_embd=2560, q_dim=4096, kv_dim=1024,
             n_ff=9728),
        # Greedy decode's vocabulary projection: logits and token.
        dict(name="head_greedy", kind="head", rows=151936, cols=2560, n_vec=1),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "session", "prefill", "prefill", "embed", "layer", "layer", "proj", "proj", "head"])
    if kind == "decode":
        shape, bf16 = rng.choice([(LLAMA, True), (QWEN, True), (GEMMA_1B, True), (GEMMA_4B, True), (GEMMA_1B, False)])
        window = rng.choice([0, 512, 1024]) if shape["head_dim"] == 256 and bf16 else 0
        return _attend(None, shape, layers=rng.randint(8, 12), pos0=_log_int(rng, 200, 32767 if bf16 else 8191), chunk=1,
                       bf16=bf16, window=window, period=6 if window else 0)
    if kind == "session":
        return _attend(None, rng.choice([LLAMA, QWEN, GEMMA_4B]), layers=rng.randint(4, 8),
                       pos0=_log_int(rng, 300, 24000), chunk=rng.randint(2, 16))
    if kind == "prefill":
        shape = rng.choice([LLAMA, QWEN, GEMMA_1B, GEMMA_4B])
        window = rng.choice([0, 512, 1024]) if shape["head_dim"] == 256 else 0
        return _attend(None, shape, layers=rng.randint(2, 4), pos0=rng.choice([0, _log_int(rng, 50, 8000)]),
                       chunk=_log_int(rng, 40, 1024), window=window, period=3 if window else 0)
    if kind == "embed":
        return _attend(None, rng.choice([EMBED, GEMMA_1B]), layers=rng.randint(2, 6), pos0=0, chunk=_log_int(rng, 60, 2048),
                       bf16=False, window=512, period=6, causal=False)
    if kind == "layer":
        shape, n_embd = rng.choice([(LLAMA, 2048), (QWEN, 2560), (GEMMA_4B, 2560)])
        n_tok = rng.choice([1, rng.randint(2, 16), _log_int(rng, 24, 512)])
        return dict(kind="layer", layers=rng.randint(2, 8) if n_tok <= 16 else 1, pos0=_log_int(rng, 200, 8000), n_tok=n_tok,
                    fmt=rng.choice(["bf16", "bf16", "q8_0", "q4_s"]), n_embd=n_embd, **shape)
    if kind == "proj":
        n_vec = rng.choice([1, 1, rng.randint(2, 16), rng.randint(2, 16), _log_int(rng, 24, 256)])
        wide = 32 * _log_int(rng, 20, 96)
        return dict(kind="proj", layers=rng.randint(3, 5) if n_vec <= 16 else 1, fmt=rng.choice(["bf16", "q8_0", "q4_s"]),
                    n_vec=n_vec, n_embd=wide, q_dim=128 * rng.randint(6, 32), kv_dim=256 * rng.randint(1, 4),
                    n_ff=32 * _log_int(rng, 36, 304))
    return dict(kind="head", rows=_log_int(rng, 32000, 152000), cols=32 * _log_int(rng, 20, 80),
                n_vec=rng.choice([1, 1, rng.randint(2, 16)]))


# ---- inputs: from the seed alone, in plain torch --------------------------------------

def _gen(seed, *path):
    s = seed & 0x7FFFFFFF
    for p in path:
        s = (s * 1000003 + p + 1) & 0x7FFFFFFFFFFF
    return torch.Generator(device=DEV).manual_seed(s)


def _randn(seed, path, *shape):
    return torch.randn(*shape, generator=_gen(seed, *path), device=DEV, dtype=torch.float32)


def _heads_normed(x, head_dim):
    h = x.view(x.shape[0], -1, head_dim)
    return (h * torch.rsqrt(h.square().mean(-1, keepdim=True) + 1e-6)).reshape(x.shape)


def _cached(case, seed, layer, n):
    """F32 K and V rows of positions 0 .. n - 1 of a layer, as the model computes them before the append."""
    d = case["n_kv"] * case["head_dim"]
    return _heads_normed(_randn(seed, (layer, 1), n, d), case["head_dim"]), _randn(seed, (layer, 2), n, d)


def _weights(seed, path, rows, cols, fmt):
    """(what the entry point takes, the same weights in 64 bits) of a random matrix in one of nnc's layouts:
    BF16, or blocks of 32 columns with a BF16 scale (and for 4 bits a BF16 bias)."""
    w = _randn(seed, path, rows, cols).mul_(1.0 / math.sqrt(cols))
    if fmt == "bf16":
        b = w.bfloat16()
        return (b,), lambda: b.double()
    blk = w.view(rows, cols // 32, 32)
    if fmt == "q8_0":
        sc = (blk.abs().amax(-1) / 127.0).bfloat16()
        q = torch.round(blk / sc.float().clamp_min(1e-30)[..., None]).clamp_(-127, 127).to(torch.int8)
        return (q.view(rows, cols), sc), lambda: (q.double() * sc.double()[..., None]).view(rows, cols)
    lo = blk.amin(-1).bfloat16()
    sc = ((blk.amax(-1) - lo.float()) / 15.0).bfloat16()
    q = torch.round((blk - lo.float()[..., None]) / sc.float().clamp_min(1e-30)[..., None]).clamp_(0, 15).to(torch.uint8)
    packed = q[..., :16] | (q[..., 16:] << 4)  # byte i of a block: elements i and i + 16
    return ((packed.reshape(rows, cols // 2).contiguous(), sc, lo),
            lambda: (q.double() * sc.double()[..., None] + lo.double()[..., None]).view(rows, cols))


def _weight_bytes(fmt, rows, cols):
    n = rows * cols
    return {"bf16": 2 * n, "q8_0": n + n // 16, "q4_s": n // 2 + n // 8}[fmt]


# ---- attention over a filled cache -------------------------------------------------------

def _window(case, layer):
    slides = case["window"] > 0 and (layer + 1) % case["period"] != 0
    return case["window"] if slides else 0


def _fill(kv, buf, k, v, rows):
    """Appends F32 rows in device memory for positions 0 .. n - 1 (those a ring keeps)."""
    lib, n = load_library(), k.shape[0]
    p = max(0, n - rows)
    while p < n:
        m = min(rows, n - p, 4096)
        if lib.nnc_hip_kv_append_f32_device(kv.handle, buf, p, m, k[p].data_ptr(), v[p].data_ptr()):
            raise RuntimeError(lib.nnc_hip_last_error().decode())
        p += m


def _prepare_attend(case, seed):
    n_tok = case["chunk"] * case["chunks"]
    n_seq = case["pos0"] + n_tok
    n_ctx = (n_seq + 255) // 256 * 256
    rows = [kv_rows(n_ctx, _window(case, li), case["chunk"]) for li in range(case["layers"])]
    kv = KVCache(rows, [case["n_kv"] * case["head_dim"]] * case["layers"], bf16=case["bf16"])
    width = case["n_head"] * case["head_dim"]
    q = torch.stack([_heads_normed(_randn(seed, (li, 0), n_tok, width), case["head_dim"]) for li in range(case["layers"])])
    for li in range(case["layers"]):
        k, v = _cached(case, seed, li, n_seq)
        torch.cuda.synchronize()
        _fill(kv, li, k, v, rows[li])
        kv.sync()
    out = torch.empty_like(q)
    torch.cuda.synchronize()
    return dict(case=case, kv=kv, q=q, out=out)


def _run_attend(s):
    c, kv, q, out = s["case"], s["kv"], s["q"], s["out"]
    step = c["chunk"] * c["n_head"] * c["head_dim"] * 4
    scale = 1.0 / math.sqrt(c["head_dim"])
    for i in range(c["chunks"]):
        for li in range(c["layers"]):
            off = (li * c["chunks"] + i) * step
            kv.attend_device(li, q.data_ptr() + off, out.data_ptr() + off, n_tok=c["chunk"], pos0=c["pos0"] + i * c["chunk"],
                             window=_window(c, li), causal=c["causal"], n_head=c["n_head"], n_kv=c["n_kv"],
                             head_dim=c["head_dim"], scale=scale)
    return out


def _spans(case, layer, pos, n_seq):
    """First and last key of positions `pos` (the last token of each call sees at most n_seq - 1)."""
    w = _window(case, layer) if "window" in case else 0
    if case.get("causal", True):
        return (torch.clamp(pos + 1 - w, min=0) if w else torch.zeros_like(pos)), pos
    if w:
        return torch.clamp(pos - w // 2, min=0), torch.clamp(pos + w // 2, max=n_seq - 1)
    return torch.zeros_like(pos), torch.full_like(pos, n_seq - 1)


def _softmax_av(q, k, v, first, last, case):
    """Attention in 64 bits: q [n, n_head * hd], k and v [n_seq, n_kv * hd], keys first .. last per row."""
    hd, g = case["head_dim"], case["n_head"] // case["n_kv"]
    n = q.shape[0]
    out = torch.empty_like(q)
    idx = torch.arange(k.shape[0], device=DEV)
    seen = (idx[None, :] >= first[:, None]) & (idx[None, :] <= last[:, None])
    for h in range(case["n_head"]):
        kh, vh = (x[:, (h // g) * hd:(h // g + 1) * hd] for x in (k, v))
        for r in range(0, n, 1024):
            s = q[r:r + 1024, h * hd:(h + 1) * hd] @ kh.t() / math.sqrt(hd)
            s.masked_fill_(~seen[r:r + 1024], -math.inf)
            out[r:r + 1024, h * hd:(h + 1) * hd] = torch.softmax(s, -1) @ vh
    return out


def _exact_attend(case, seed):
    n_tok = case["chunk"] * case["chunks"]
    n_seq = case["pos0"] + n_tok
    pos = torch.arange(case["pos0"], n_seq, device=DEV)
    got = []
    for li in range(case["layers"]):
        q = _heads_normed(_randn(seed, (li, 0), n_tok, case["n_head"] * case["head_dim"]), case["head_dim"]).double()
        k, v = _cached(case, seed, li, n_seq)
        if case["bf16"]:
            k, v = k.bfloat16(), v.bfloat16()
        got.append(_softmax_av(q, k.double(), v.double(), *_spans(case, li, pos, n_seq), case))
    return torch.stack(got)


def _attend_work(case):
    n_tok = case["chunk"] * case["chunks"]
    b = f = 0
    for li in range(case["layers"]):
        for i in range(case["chunks"]):
            p0 = case["pos0"] + i * case["chunk"]
            pos = torch.arange(p0, p0 + case["chunk"])
            first, last = _spans(case, li, pos, p0 + case["chunk"])
            f += 4 * case["head_dim"] * case["n_head"] * int((last - first + 1).sum())
            b += 2 * int(last[-1] - first[0] + 1) * case["n_kv"] * case["head_dim"] * (2 if case["bf16"] else 4)
    b += 2 * case["layers"] * n_tok * case["n_head"] * case["head_dim"] * 4
    return dict(bytes=b, flops=f)


# ---- the attention half of a layer ---------------------------------------------------------

ROPE_BASE = 1000000.0


def _layer_dims(case):
    return case["n_head"] * case["head_dim"], case["n_kv"] * case["head_dim"]


def _layer_inputs(case, seed, li):
    qd, kd = _layer_dims(case)
    e, hd, fmt = case["n_embd"], case["head_dim"], case["fmt"]
    mats = [_weights(seed, (li, 10 + j), r, c, fmt) for j, (r, c) in enumerate([(qd, e), (kd, e), (kd, e), (e, qd)])]
    gam = [1.0 + 0.1 * _randn(seed, (li, 20 + j), hd) for j in range(2)]
    return mats, gam, _randn(seed, (li, 30), case["n_tok"], e)


def _prepare_layer(case, seed):
    qd, kd = _layer_dims(case)
    n, e = case["n_tok"], case["n_embd"]
    n_seq = case["pos0"] + n
    kv = KVCache([(n_seq + 255) // 256 * 256] * case["layers"], [kd] * case["layers"], bf16=True)
    ws, gs, xs, preps = [], [], [], []
    for li in range(case["layers"]):
        mats, gam, x = _layer_inputs(case, seed, li)
        k, v = _cached(case, seed, li, case["pos0"])
        torch.cuda.synchronize()
        _fill(kv, li, k, v, n_seq)
        kv.sync()
        ws.append([m[0] for m in mats])
        gs.append(gam)
        xs.append(x)
        preps.append(NncHipPrep(case["n_head"], case["n_kv"], case["head_dim"], gam[0].data_ptr(), gam[1].data_ptr(), 0,
                                1e-6, case["head_dim"], ROPE_BASE, 1.0, 0, None))
    f32 = dict(device=DEV, dtype=torch.float32)
    s = dict(case=case, kv=kv, w=ws, g=gs, x=xs, prep=preps, q=torch.empty(case["layers"], n, qd, **f32),
             k=torch.empty(n, kd, **f32), v=torch.empty(n, kd, **f32), a=torch.empty(n, qd, **f32),
             out=torch.empty(case["layers"], n, e, **f32))
    torch.cuda.synchronize()
    return s


def _addr(w):
    return tuple(t.data_ptr() for t in w)


def _run_layer(s):
    c, kv = s["case"], s["kv"]
    qd, kd = _layer_dims(c)
    n, e = c["n_tok"], c["n_embd"]
    k, v, a = s["k"].data_ptr(), s["v"].data_ptr(), s["a"].data_ptr()
    for li in range(c["layers"]):
        w, q = s["w"][li], s["q"].data_ptr() + li * n * qd * 4
        kv.gemv_group_device(c["fmt"], [(_addr(w[0]), q, qd), (_addr(w[1]), k, kd), (_addr(w[2]), v, kd)],
                             s["x"][li].data_ptr(), cols=e, n_batch=n)
        kv.prep_append_device(li, q, k, v, pos0=c["pos0"], n_tok=n, prep=s["prep"][li])
        kv.attend_device(li, q, a, n_tok=n, pos0=c["pos0"], n_head=c["n_head"], n_kv=c["n_kv"], head_dim=c["head_dim"],
                         scale=1.0 / math.sqrt(c["head_dim"]))
        kv.gemv_device(c["fmt"], _addr(w[3]), a, s["out"].data_ptr() + li * n * e * 4, rows=e, cols=qd, n_batch=n)
    return {"q": s["q"], "out": s["out"]}


def _rope64(x, pos0, hd):
    """NEOX rotation in 64 bits at the model's angles, which are formed in 32 bits by definition."""
    ratio = np.float32(float(ROPE_BASE) ** float(np.float32(-2.0 / hd)))
    inv, f = [], np.float32(1.0)
    for _ in range(hd // 2):
        inv.append(f)
        f = np.float32(f * ratio)
    th = np.arange(pos0, pos0 + x.shape[0], dtype=np.float32)[:, None] * np.array(inv, np.float32)[None, :]
    th = torch.from_numpy(th.astype(np.float64)).to(DEV)[:, None, :]
    h = x.view(x.shape[0], -1, hd)
    a, b = h[..., :hd // 2], h[..., hd // 2:]
    return torch.cat([a * th.cos() - b * th.sin(), a * th.sin() + b * th.cos()], -1).reshape(x.shape)


def _exact_layer(case, seed):
    hd, n = case["head_dim"], case["n_tok"]
    pos = torch.arange(case["pos0"], case["pos0"] + n, device=DEV)
    qs, outs = [], []
    for li in range(case["layers"]):
        mats, gam, x = _layer_inputs(case, seed, li)
        x = x.double()
        q, k, v = (x @ m[1]().t() for m in mats[:3])
        for_head = lambda y, g: ((y.view(n, -1, hd) * torch.rsqrt(y.view(n, -1, hd).square().mean(-1, keepdim=True) + 1e-6))
                                 * g.double()).reshape(y.shape)  # noqa: E731
        q, k = (_rope64(for_head(y, g), case["pos0"], hd) for y, g in zip((q, k), gam))
        ck, cv = _cached(case, seed, li, case["pos0"])
        k, v = (torch.cat([c.bfloat16().double(), y.float().bfloat16().double()]) for c, y in ((ck, k), (cv, v)))
        a = _softmax_av(q, k, v, torch.zeros_like(pos), pos, case)
        qs.append(q)
        outs.append(a @ mats[3][1]().t())
    return {"q": torch.stack(qs), "out": torch.stack(outs)}


def _layer_work(case):
    qd, kd = _layer_dims(case)
    e, n, p, fmt = case["n_embd"], case["n_tok"], case["pos0"], case["fmt"]
    w = _weight_bytes(fmt, qd, e) + 2 * _weight_bytes(fmt, kd, e) + _weight_bytes(fmt, e, qd)
    b = w + 4 * n * (e + e + qd) + 2 * (p + n) * kd * 2
    f = 2 * n * e * (2 * qd + 2 * kd) + 4 * qd * (n * p + n * (n + 1) // 2)
    return dict(bytes=case["layers"] * b, flops=case["layers"] * f)


# ---- weight products -------------------------------------------------------------------------

def _proj_groups(case):
    """(input width, rows of the matrices that share the input) per launch of a layer."""
    e, q, k, f = (case[x] for x in ("n_embd", "q_dim", "kv_dim", "n_ff"))
    return [(e, (q, k, k)), (q, (e,)), (e, (f, f)), (f, (e,))]


def _proj_inputs(case, seed, li):
    return [([_weights(seed, (li, gi, j), r, cols, case["fmt"]) for j, r in enumerate(rows)],
             _randn(seed, (li, gi, 9), case["n_vec"], cols)) for gi, (cols, rows) in enumerate(_proj_groups(case))]


def _prepare_proj(case, seed):
    kv = KVCache([16], [64])
    total = sum(sum(rows) for _, rows in _proj_groups(case)) * case["n_vec"]
    layers = [[([m[0] for m in mats], x) for mats, x in _proj_inputs(case, seed, li)] for li in range(case["layers"])]
    y = torch.empty(case["layers"], total, device=DEV, dtype=torch.float32)
    torch.cuda.synchronize()
    return dict(case=case, kv=kv, layers=layers, y=y)


def _run_proj(s):
    c, kv = s["case"], s["kv"]
    n, at = c["n_vec"], s["y"].data_ptr()
    for layer in s["layers"]:
        for (cols, rows), (ws, x) in zip(_proj_groups(c), layer):
            ys = []
            for r in rows:
                ys.append(at)
                at += 4 * n * r
            if len(rows) == 1:
                kv.gemv_device(c["fmt"], _addr(ws[0]), x.data_ptr(), ys[0], rows=rows[0], cols=cols, n_batch=n)
            else:
                kv.gemv_group_device(c["fmt"], [(_addr(w), y, r) for w, y, r in zip(ws, ys, rows)], x.data_ptr(), cols=cols,
                                     n_batch=n)
    return s["y"]


def _exact_proj(case, seed):
    return torch.stack([torch.cat([(x.double() @ m[1]().t()).reshape(-1) for mats, x in _proj_inputs(case, seed, li)
                                   for m in mats]) for li in range(case["layers"])])


def _proj_work(case):
    b = f = 0
    for cols, rows in _proj_groups(case):
        b += sum(_weight_bytes(case["fmt"], r, cols) for r in rows) + 4 * case["n_vec"] * (cols + sum(rows))
        f += 2 * case["n_vec"] * cols * sum(rows)
    return dict(bytes=case["layers"] * b, flops=case["layers"] * f)


# ---- the vocabulary projection ---------------------------------------------------------------

def _head_inputs(case, seed):
    return _weights(seed, (0,), case["rows"], case["cols"], "bf16"), _randn(seed, (1,), case["n_vec"], case["cols"])


def _prepare_head(case, seed):
    kv = KVCache([16], [64])
    (w, _), x = _head_inputs(case, seed)
    y = torch.empty(case["n_vec"], case["rows"], device=DEV, dtype=torch.float32)
    torch.cuda.synchronize()
    return dict(case=case, kv=kv, w=w, x=x, y=y)


def _run_head(s):
    c, kv = s["case"], s["kv"]
    kv.gemv_device("bf16", _addr(s["w"]), s["x"].data_ptr(), s["y"].data_ptr(), rows=c["rows"], cols=c["cols"],
                   n_batch=c["n_vec"])
    if c["n_vec"] > 1:
        return {"logits": s["y"]}
    token = kv.gemv_argmax_device(s["w"][0].data_ptr(), s["x"].data_ptr(), rows=c["rows"], cols=c["cols"])
    return {"logits": s["y"], "token": token}


def _exact_head(case, seed):
    (_, w64), x = _head_inputs(case, seed)
    y = x.double() @ w64().t()
    return {"logits": y, "token": int(y[0].argmax())} if case["n_vec"] == 1 else {"logits": y}


def _head_work(case):
    calls = 2 if case["n_vec"] == 1 else 1  # the greedy token is a call of its own
    return dict(bytes=calls * 2 * case["rows"] * case["cols"] + 4 * case["n_vec"] * (case["rows"] + calls * case["cols"]),
                flops=calls * 2 * case["n_vec"] * case["rows"] * case["cols"])


_KINDS = {"attend": (_prepare_attend, _run_attend, _attend_work, _exact_attend),
          "layer": (_prepare_layer, _run_layer, _layer_work, _exact_layer),
          "proj": (_prepare_proj, _run_proj, _proj_work, _exact_proj),
          "head": (_prepare_head, _run_head, _head_work, _exact_head)}


def prepare(case, seed):
    return _KINDS[case["kind"]][0](case, seed)


def run(state):
    return _KINDS[state["case"]["kind"]][1](state)


def work(case):
    return _KINDS[case["kind"]][2](case)


def exact(case, seed):
    return _KINDS[case["kind"]][3](case, seed)


def tolerance(case):
    """Relative error in the 2-norm, about four times what the paths measure against exact()."""
    n = case.get("n_tok", case.get("chunk", 1))
    if case["kind"] == "attend" and not case["bf16"]:
        return {"rel": 2e-5}  # 32-bit sums; decode splits q and k into two 16-bit halves (4e-6)
    if case["kind"] in ("attend", "layer") and n > 16:
        return {"rel": 8e-4}  # weights of the long batches' P . V product in 16 bits (2e-4)
    if case["kind"] == "layer":
        return {"rel": 5e-5}  # 3e-6, and a K or V element now and then on the other side of a BF16 rounding
    # q, and activations of batches, as two 16-bit halves, 32-bit sums (3e-6; one vector's products 3e-7)
    return {"rel": 2e-5} if case["kind"] == "attend" else {"rel": 1e-5}
