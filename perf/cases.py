"""The work that users of the verify path have it do, as cases to time.

A case is a dict of plain values.  `prepare` makes what a program holds before
the call (weights in the kernels' tiled layout, a paged KV cache, inputs, and
the captured graph where such a program replays one), `run` is one pass through
the public entry points, `exact` the same result in 64 bits by plain torch.

Kinds of case, by entry point:
  step       opure_verify_step of a whole model: one speculative step with
             greedy acceptance and rollback, replayed from its graph
  prompt     opure_engine_forward_logits: a whole prompt prefilled, the last
             position's logits back on the host
  layer      opure_verify_layer on a residual: one sequence's K+1 rows, a batch
             of sequences with ragged contexts (both replayed from a graph), or
             a 16-row-parts chunk of one prompt as the engine's prefill makes it
  attention  opure_attn_decode_paged alone, any head size, ragged contexts
  gemv       opure_gemv_batched_* alone
  reject     opure_accept_rejection: rejection sampling over stored logits
  sample     opure_sample_rows: drafting at a temperature
  greedy     opure_accept_greedy over stored logits

All GPU work of a process goes through one device handle, so passes on
different states queue on one stream as a program's would.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "opure-voxelengine_amd"))
import opure_engine as E  # noqa: E402
import opure_hip as H  # noqa: E402

PAGE = H.PAGE_SIZE
WFMT = {"f32": H.W_F32, "i8": H.W_I8PC, "i4": H.W_I4G128}
AFMT = {"f32": H.A_F32, "f16": H.A_F16, "bf16": H.A_BF16}
DTYPE = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
KBLOCK = {"f32": 16, "i8": 64, "i4": 128}
GEMV = {"f32": "opure_gemv_batched_f32", "i8": "opure_gemv_batched_i8pc", "i4": "opure_gemv_batched_i4g128"}

# model shapes: the three that the benchmark's configurations name
SMOL = dict(hidden=576, heads=9, kv=3, hd=64, ffn=1536, w="f32", a="f32")
ONE_B = dict(hidden=2048, heads=32, kv=8, hd=64, ffn=8192, w="i8", a="f16")
EIGHT_B = dict(hidden=4096, heads=32, kv=8, hd=128, ffn=14336, w="i4", a="bf16")


def listed():
    return [
        # the headline use: a speculative step of a 1B model, 5 drafts, 2k context
        dict(name="step 1b int8", kind="step", **ONE_B, layers=16, vocab=128256, batch=1, rows=6, ctx=2048, ragged=0),
        # a new request: its whole prompt through the engine, an odd length
        dict(name="prompt 1b int8", kind="prompt", **ONE_B, layers=16, vocab=128256, tokens=1437),
        # the smallest model that is served: a layer at a short context, fp32 throughout
        dict(name="layer 135m f32", kind="layer", **SMOL, mode="verify", batch=1, rows=5, ctx=300, ragged=0),
        # a large model's layer at a long context, 7 drafts
        dict(name="layer 8b int4 bf16", kind="layer", **EIGHT_B, mode="verify", batch=1, rows=8, ctx=8000, ragged=0),
        # a server's batch: 32 sequences with 6 drafts each, contexts from 512 to 8192
        dict(name="layer 1b int8 batch", kind="layer", **ONE_B, mode="verify", batch=32, rows=7, ctx=8185, ragged=512),
        # a server's batch without drafts: one new token for each of 24 sequences
        dict(name="layer 8b int4 f16 decode", kind="layer", **{**EIGHT_B, "a": "f16"}, mode="verify", batch=24, rows=1,
             ctx=4001, ragged=200),
        # a chunk of a long prompt through a large model's layer, as the engine's prefill launches it
        dict(name="layer 8b int4 prompt", kind="layer", **EIGHT_B, mode="prompt", batch=16, rows=16, ctx=1024, ragged=0),
        # attention of a model whose heads are neither 64 nor 128 wide
        dict(name="attention hd96 f16", kind="attention", heads=32, kv=8, hd=96, a="f16", batch=4, rows=5, ctx=1500,
             ragged=100),
        # the smallest call there is: one row through one small linear
        dict(name="gemv 576 f32", kind="gemv", out=576, inn=576, w="f32", a="f32", rows=1, swiglu=False),
        # rejection sampling of a large batch
        dict(name="reject 64x8 49k", kind="reject", batch=64, k=8, vocab=49152, temperature=1.0, near=0.0),
        # drafts drawn at a temperature, a large vocabulary
        dict(name="sample 16 128k", kind="sample", rows=16, vocab=128256, temperature=0.8),
        # greedy acceptance over logits that a program already has
        dict(name="greedy 16x5 128k", kind="greedy", batch=16, k=5, vocab=128256),
    ]


def _log(rng, lo, hi):
    """A whole number spread evenly over the logarithm of lo..hi."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_model(rng):
    w = rng.choice(["f32", "i8", "i8", "i4", "i4", "i4"])
    if w == "f32":
        kv = rng.randint(2, 5)
        heads = kv * rng.choice([1, 2, 3])
        return dict(hidden=heads * 64, heads=heads, kv=kv, hd=64, ffn=64 * rng.randint(8, 40), w="f32", a="f32")
    if w == "i8":
        hd = rng.choice([64, 64, 128])
        kv = rng.choice([4, 8])
        heads = kv * rng.randint(2, 4) if hd == 64 else kv * 2
        return dict(hidden=128 * rng.randint(6, 20), heads=heads, kv=kv, hd=hd, ffn=64 * rng.randint(40, 144), w="i8",
                    a="f16")
    hd = rng.choice([64, 128, 128])
    heads = 8 * rng.randint(2, 4)
    return dict(hidden=128 * rng.randint(12, 34), heads=heads, kv=8, hd=hd, ffn=128 * rng.randint(32, 112), w="i4",
                a=rng.choice(["f16", "bf16"]))


def draw(rng):
    """One more case of the listed ones' ranges: the same entry points, formats
    and options, sizes up to the listed largest, odd ones among them."""
    kind = rng.choice(["layer"] * 8 + ["attention"] * 3 + ["gemv"] * 3 + ["step", "prompt", "reject", "reject", "sample",
                                                                         "greedy"])
    if kind in ("layer", "step", "prompt"):
        m = _draw_model(rng)
        if kind == "prompt":
            if m["w"] == "f32":
                m = dict(ONE_B)
            return dict(kind=kind, **m, layers=rng.randint(1, 4), vocab=16 * _log(rng, 500, 4000), tokens=_log(rng, 20, 3000))
        if kind == "step":
            rows = rng.randint(1, 9)
            ctx = PAGE * _log(rng, 2, 400) + rng.randint(0, PAGE - rows)
            return dict(kind=kind, **m, layers=rng.randint(1, 4), vocab=16 * _log(rng, 500, 8016), batch=1, rows=rows,
                        ctx=ctx if m["w"] != "f32" else ctx % 2000, ragged=0)
        mode = rng.choice(["one", "batch", "batch", "prompt"]) if m["w"] != "f32" else "one"
        if mode == "one":
            ctx = _log(rng, 16, 8192) if m["w"] != "f32" else _log(rng, 16, 2000)
            return dict(kind=kind, **m, mode="verify", batch=1, rows=rng.randint(1, 9), ctx=ctx, ragged=0)
        if mode == "batch":
            rows = rng.choice([1, 1, rng.randint(2, 8)])
            ctx = _log(rng, 256, 6000)
            return dict(kind=kind, **m, mode="verify", batch=min(_log(rng, 2, 64), 256 // rows), rows=rows, ctx=ctx,
                        ragged=max(8, ctx // rng.randint(2, 16)))
        return dict(kind=kind, **m, mode="prompt", batch=rng.randint(2, 16), rows=16, ctx=16 * rng.randint(0, 250), ragged=0)
    if kind == "attention":
        kv = rng.choice([2, 4, 8])
        hd = rng.choice([32, 48, 64, 64, 80, 96, 112, 128, 128, 160, 192, 256])
        ctx = _log(rng, 64, 6000)
        return dict(kind=kind, heads=kv * rng.randint(1, 4), kv=kv, hd=hd, a=rng.choice(["f16", "bf16", "f16", "f32"]),
                    batch=_log(rng, 1, 12), rows=rng.randint(1, 8), ctx=ctx, ragged=max(8, ctx // rng.randint(1, 16)))
    if kind == "gemv":
        w = rng.choice(["f32", "i8", "i4", "i4"])
        kb = KBLOCK[w]
        out, inn = 32 * _log(rng, 8, 1000), kb * max(1, _log(rng, 256, 14336) // kb)
        if w == "f32":
            inn = min(inn, 4096)
        return dict(kind=kind, out=out, inn=inn, w=w, a={"f32": "f32", "i8": "f16"}.get(w) or rng.choice(["f16", "bf16"]),
                    rows=_log(rng, 1, 16 if w == "f32" else 256), swiglu=rng.random() < 0.3)
    vocab = 16 * _log(rng, 500, 8016) + rng.choice([0, 0, 1, 7])
    if kind == "sample":
        return dict(kind=kind, rows=_log(rng, 1, 64), vocab=vocab, temperature=rng.choice([0.3, 0.7, 0.8, 1.0]))
    if kind == "greedy":
        return dict(kind=kind, batch=_log(rng, 1, 32), k=rng.randint(1, 8), vocab=vocab)
    return dict(kind=kind, batch=_log(rng, 1, 32), k=rng.randint(1, 8), vocab=vocab,
                temperature=rng.choice([0.6, 0.8, 1.0]), near=rng.choice([0.0, 0.5, 0.9]))


# ---- inputs ------------------------------------------------------------------

_dev = None


def _device():
    """The one device handle of the process, as a program has it."""
    global _dev
    if _dev is None:
        torch.zeros(1, device="cuda")
        _dev = H.Dev(torch.cuda.current_device())
    return _dev


def _gen(seed, salt):
    return torch.Generator("cuda").manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFFFFFF)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _linear(g, out, inn, w, std=0.02):
    """A linear in the row-major interchange form: N(0, std) weights, quantised."""
    x = _randn(g, out, inn).mul_(std)
    if w == "f32":
        return dict(w=x, out=out, inn=inn, fmt=w)
    if w == "i8":
        s = (x.abs().amax(1, keepdim=True) / 127).half()
        q = (x / s.float()).round_().clamp_(-127, 127).to(torch.int8)
        return dict(w=q, scale=s.reshape(-1).contiguous(), out=out, inn=inn, fmt=w)
    x = x.reshape(out, inn // 128, 128)
    lo, hi = x.amin(2, keepdim=True), x.amax(2, keepdim=True)
    s = ((hi - lo) / 15).bfloat16()
    z = (-lo / s.float()).bfloat16()
    q = (x / s.float() + z.float()).round_().clamp_(0, 15).to(torch.uint8).reshape(out, inn // 2, 2)
    return dict(w=(q[:, :, 0] << 4) | q[:, :, 1], scale=s.squeeze(2).contiguous(), zero=z.squeeze(2).contiguous(),
                out=out, inn=inn, fmt=w)


def _dense(d):
    """The linear's values in 64 bits."""
    if d["fmt"] == "f32":
        return d["w"].double()
    if d["fmt"] == "i8":
        return d["w"].double() * d["scale"].double()[:, None]
    q = torch.stack((d["w"] >> 4, d["w"] & 15), 2).reshape(d["out"], -1, 128).double()
    return ((q - d["zero"].double()[:, :, None]) * d["scale"].double()[:, :, None]).reshape(d["out"], d["inn"])


def _layer_weights(case, seed, layer):
    g = _gen(seed, 100 + layer)
    h, qd, kd, w = case["hidden"], case["heads"] * case["hd"], case["kv"] * case["hd"], case["w"]
    return dict(qkv=_linear(g, qd + 2 * kd, h, w), o=_linear(g, h, qd, w), gate_up=_linear(g, 2 * case["ffn"], h, w),
                down=_linear(g, h, case["ffn"], w), attn_norm=1 + 0.1 * _randn(g, h), mlp_norm=1 + 0.1 * _randn(g, h))


def _head_weights(case, seed):
    """The embedding, which is the LM head too.  Rows are longer than the other
    weights', so a token's own logit stands out as a trained model's choice does."""
    g = _gen(seed, 1)
    return _linear(g, case["vocab"], case["hidden"], case["w"], 0.5), 1 + 0.1 * _randn(g, case["hidden"])


THETA = 500000.0


def _contexts(case):
    """Cached tokens of each sequence: a ragged batch spreads from ragged to ctx
    evenly over the logarithm, in no order; a prompt's parts follow each other."""
    n = case["batch"]
    if case.get("mode") == "prompt":
        return [case["ctx"] + PAGE * i for i in range(n)]
    if not case["ragged"] or n == 1:
        return [case["ctx"]] * n
    lens = [round(case["ragged"] * (case["ctx"] / case["ragged"]) ** (i / (n - 1))) for i in range(n)]
    return [lens[i] for i in np.random.RandomState(n).permutation(n)]


def _cache(case, seed, layers):
    """A paged KV cache filled to the contexts, in pages taken in no order; the
    pages that the call appends to come first in the pool, so that one view holds them."""
    g = _gen(seed, 2)
    lens, rows, shared = _contexts(case), case["rows"], case.get("mode") == "prompt"
    seqs = [(lens[0], lens[-1] + rows)] if shared else [(n, n + rows) for n in lens]
    tails = [list(range(a // PAGE, (b + PAGE - 1) // PAGE)) for a, b in seqs]
    n_tail = sum(len(t) for t in tails)
    n_pages = sum((b + PAGE - 1) // PAGE for _, b in seqs)
    cols = max((b + PAGE - 1) // PAGE for _, b in seqs)
    order = (torch.randperm(n_pages - n_tail, generator=torch.Generator().manual_seed(int(seed) + 5)) + n_tail).tolist()
    table = np.full((case["batch"], cols), -1, np.int32)
    used = at = 0
    for i, (_, b) in enumerate(seqs):
        for j in range((b + PAGE - 1) // PAGE):
            if j in tails[i]:
                table[i, j], used = used, used + 1
            else:
                table[i, j], at = order[at], at + 1
    if shared:
        table[:] = table[0]
    pool = torch.randn(layers, n_pages, 2, case["kv"], PAGE * case["hd"], generator=g, device="cuda", dtype=DTYPE[case["a"]])
    return dict(pool=pool, table=table, lens=lens, n_tail=n_tail, n_pages=n_pages, cols=cols,
                max_ctx=max(lens) + rows)


def _tokens(case, seed):
    """The last token, the drafts that the target will take, and one that it will not."""
    r = np.random.RandomState((int(seed) * 7 + 3) & 0x7FFFFFFF)
    t = np.full((case["batch"], case["rows"]), 0, np.int32)
    for b in range(case["batch"]):
        t[b, :] = r.randint(case["vocab"])
        if case["rows"] > 2:
            t[b, -1] = (t[b, 0] + 1) % case["vocab"]
    return t


def _logits(g, rows, vocab):
    return _randn(g, rows, vocab).mul_(3.0)


# ---- device state --------------------------------------------------------------


class State:
    """What a program holds: device buffers, descriptors, and a graph where it has one."""

    def __init__(self):
        self.keep, self.graph, self.engine, self.call, self.out = [], None, None, None, None

    def ptr(self, t):
        self.keep.append(t)
        return t.data_ptr()

    def __del__(self):
        if self.engine is not None:
            self.engine.close()
        if self.graph is not None:
            _device().graph_destroy(self.graph)


def _tiled(st, d, swiglu=False):
    dev, w = _device(), WFMT[d["fmt"]]
    wb, sb = C.c_uint64(), C.c_uint64()
    H.check(H.lib().opure_tiled_bytes(w, d["out"], d["inn"], C.byref(wb), C.byref(sb)))
    dst_w = torch.empty(wb.value, dtype=torch.uint8, device="cuda")
    dst_s = torch.empty(max(1, sb.value), dtype=torch.uint8, device="cuda")
    src = H.Linear(d["w"].data_ptr(), d["scale"].data_ptr() if "scale" in d else None,
                   d["zero"].data_ptr() if "zero" in d else None, d["out"], d["inn"], H.LAYOUT_ROWMAJOR)
    dst = H.Linear()
    torch.cuda.synchronize()
    H.check(H.lib().opure_tile_linear(dev.h, w, H.LAYOUT_TILED_SWIGLU if swiglu else H.LAYOUT_TILED, C.byref(src),
                                      st.ptr(dst_w), st.ptr(dst_s), C.byref(dst)))
    dev.sync()
    return dst


def _model(st, case, seed, layers, max_pos, head=None):
    """opure_model of the case's weights; `head`: the embedding and final gain (a layer alone has none)."""
    lw = (H.LayerWeights * layers)()
    for i in range(layers):
        d = _layer_weights(case, seed, i)
        lw[i] = H.LayerWeights(st.ptr(d["attn_norm"]), st.ptr(d["mlp_norm"]), _tiled(st, d["qkv"]), _tiled(st, d["o"]),
                               _tiled(st, d["gate_up"], True), _tiled(st, d["down"]))
    st.keep.append(lw)
    emb, gain = head if head is not None else (_linear(_gen(seed, 1), 16, case["hidden"], case["w"]),
                                               torch.ones(case["hidden"], device="cuda"))
    e = _tiled(st, emb)
    cos, sin = (torch.from_numpy(t).cuda() for t in H.rope_table(THETA, case["hd"], max_pos, H.ROPE_GPU))
    m = H.Model(layers, case["hidden"], case["heads"], case["kv"], case["hd"], case["ffn"], emb["out"], 1e-5,
                case["hd"] ** -0.5, WFMT[case["w"]], AFMT[case["a"]], st.ptr(cos), st.ptr(sin), max_pos, e, e,
                st.ptr(gain), C.cast(lw, C.POINTER(H.LayerWeights)))
    st.keep.append(m)
    return m


def _kv(st, cache):
    table = torch.from_numpy(cache["table"]).cuda()
    kv = H.KV(st.ptr(cache["pool"]), cache["n_pages"], PAGE, st.ptr(table), cache["cols"])
    st.keep.append(kv)
    st.lens = torch.tensor(cache["lens"], dtype=torch.int32, device="cuda")
    return kv


def _capture(st, call):
    """The call recorded once; a pass replays it."""
    dev = _device()
    call()
    dev.sync()
    dev.graph_begin()
    call()
    st.graph = dev.graph_end()


def _prepare_step(case, seed):
    st, dev = State(), _device()
    cache = _cache(case, seed, case["layers"])
    m = _model(st, case, seed, case["layers"], cache["max_ctx"], _head_weights(case, seed))
    kv = _kv(st, cache)
    B, R = case["batch"], case["rows"]
    tok = torch.from_numpy(_tokens(case, seed)).cuda()
    logits = torch.empty(B, R, case["vocab"], device="cuda")
    ints = [torch.empty(*s, dtype=torch.int32, device="cuda") for s in ((B, R), (B,), (B,))]
    a = H.VerifyArgs()
    a.model, a.kv, a.batch, a.rows = C.pointer(m), C.pointer(kv), B, R
    a.tokens, a.seq_len, a.max_ctx, a.logits = st.ptr(tok), st.ptr(st.lens), cache["max_ctx"], st.ptr(logits)
    a.accept_mode, a.temperature = H.ACCEPT_GREEDY, 1.0
    a.out_tokens, a.accepted, a.rollback, a.new_seq_len = (st.ptr(ints[0]), st.ptr(ints[1]), 1, st.ptr(ints[2]))
    torch.cuda.synchronize()
    H.check(H.lib().opure_verify_reserve(dev.h, C.byref(m), B, R, cache["max_ctx"]))
    _capture(st, lambda: H.check(H.lib().opure_verify_step(dev.h, C.byref(a))))
    st.keep.append(a)
    st.out = dict(logits=logits, tokens=ints[0], accepted=ints[1], length=ints[2], kv=cache["pool"][:, :cache["n_tail"]])
    return st


def _prepare_prompt(case, seed):
    st, dev = State(), _device()
    r = np.random.RandomState((int(seed) * 7 + 3) & 0x7FFFFFFF)
    st.tokens, st.vocab = r.randint(case["vocab"], size=case["tokens"]).astype(np.int32), case["vocab"]
    m = _model(st, case, seed, case["layers"], 4096, _head_weights(case, seed))
    torch.cuda.synchronize()
    st.engine = E.Engine(dev, m, None, 4096)
    return st


def _prepare_layer(case, seed):
    st, dev = State(), _device()
    cache = _cache(case, seed, 1)
    m = _model(st, case, seed, 1, cache["max_ctx"])
    kv = _kv(st, cache)
    B, R = case["batch"], case["rows"]
    st.x0 = _randn(_gen(seed, 3), B * R, case["hidden"])
    st.x = st.x0.clone()
    a = H.VerifyLayerArgs(C.pointer(m), C.pointer(kv), 0, B, R, st.ptr(st.lens), cache["max_ctx"], st.x.data_ptr())
    torch.cuda.synchronize()
    H.check(H.lib().opure_verify_reserve(dev.h, C.byref(m), B, R, cache["max_ctx"]))
    L, ref, x, x0, n = H.lib(), C.byref(a), st.x.data_ptr(), st.x0.data_ptr(), st.x.numel() * 4

    def call():
        # the layer works in place: its input comes from the layer before
        H.check(L.opure_buf_copy(dev.h, x, x0, n))
        H.check(L.opure_verify_layer(dev.h, ref))

    st.keep.append(a)
    if case["mode"] == "prompt":
        st.call = call            # a prompt's chunks are launched one by one
    else:
        _capture(st, call)
    st.out = dict(x=st.x, kv=cache["pool"][:, :cache["n_tail"]])
    return st


def _prepare_attention(case, seed):
    st, dev = State(), _device()
    cache = _cache(case, seed, 1)
    kv = _kv(st, cache)
    B, R = case["batch"], case["rows"]
    q = _randn(_gen(seed, 3), B * R, case["heads"] * case["hd"]).to(DTYPE[case["a"]])
    out = torch.empty_like(q)
    m = H.Model()
    m.n_layers, m.n_heads, m.n_kv_heads, m.head_dim = 1, case["heads"], case["kv"], case["hd"]
    m.attn_scale, m.afmt = case["hd"] ** -0.5, AFMT[case["a"]]
    st.keep.append(m)
    a = H.AttnArgs(C.pointer(m), C.pointer(kv), 0, B, R, st.ptr(st.lens), cache["max_ctx"], st.ptr(q), st.ptr(out))
    L, ref = H.lib(), C.byref(a)
    st.keep.append(a)
    st.call = lambda: H.check(L.opure_attn_decode_paged(dev.h, ref))
    st.out = out
    return st


def _gemv_inputs(case, seed):
    d = _linear(_gen(seed, 1), case["out"], case["inn"], case["w"])
    return d, _randn(_gen(seed, 3), case["rows"], case["inn"]).to(DTYPE[case["a"]])


def _prepare_gemv(case, seed):
    st, dev = State(), _device()
    d, x = _gemv_inputs(case, seed)
    lin = _tiled(st, d, case["swiglu"])
    y = torch.empty(case["rows"], case["out"] // (2 if case["swiglu"] else 1), device="cuda", dtype=DTYPE[case["a"]])
    a = H.GemvArgs(lin, st.ptr(x), st.ptr(y), case["rows"], AFMT[case["a"]], AFMT[case["a"]],
                   H.EPI_SWIGLU if case["swiglu"] else H.EPI_STORE)
    fn, ref = getattr(H.lib(), GEMV[case["w"]]), C.byref(a)
    st.keep.append(a)
    st.call = lambda: H.check(fn(dev.h, ref))
    st.out = y
    return st


def _reject_inputs(case, seed):
    """Target and draft logits (the draft model follows the target by `near`) and
    drafts drawn from the draft's distribution."""
    g = _gen(seed, 3)
    B, K, V = case["batch"], case["k"], case["vocab"]
    t = _logits(g, B * (K + 1), V).reshape(B, K + 1, V)
    q = t[:, :K] * case["near"] + _logits(g, B * K, V).reshape(B, K, V) * math.sqrt(1 - case["near"] ** 2)
    q = q.contiguous()
    race = torch.empty(B, K, V, device="cuda").exponential_(generator=g).log_().neg_()
    return t, q, (q / case["temperature"] + race).argmax(2).to(torch.int32).contiguous()


def _prepare_reject(case, seed):
    st, dev = State(), _device()
    t, q, d = _reject_inputs(case, seed)
    B, K, V = case["batch"], case["k"], case["vocab"]
    tok = torch.empty(B, K + 1, dtype=torch.int32, device="cuda")
    acc = torch.empty(B, dtype=torch.int32, device="cuda")
    dist = torch.empty(B, V, device="cuda")
    a = H.AcceptArgs(B, K, V, st.ptr(t), st.ptr(q), st.ptr(d), K, case["temperature"], int(seed), None, st.ptr(tok),
                     st.ptr(acc), st.ptr(dist))
    L, ref = H.lib(), C.byref(a)
    st.keep.append(a)
    st.call = lambda: H.check(L.opure_accept_rejection(dev.h, ref))
    st.out = dict(tokens=tok, accepted=acc, dist=dist)
    return st


def _prepare_sample(case, seed):
    st, dev = State(), _device()
    n = case["rows"]
    lg = _logits(_gen(seed, 3), n, case["vocab"])
    pos = torch.full((n,), 77, dtype=torch.int32, device="cuda")
    seq = torch.arange(n, dtype=torch.int32, device="cuda")
    out = torch.empty(n, dtype=torch.int32, device="cuda")
    a = H.SampleArgs(n, case["vocab"], st.ptr(lg), case["temperature"], int(seed), st.ptr(pos), st.ptr(seq), 0, st.ptr(out))
    L, ref = H.lib(), C.byref(a)
    st.keep.append(a)
    st.call = lambda: H.check(L.opure_sample_rows(dev.h, ref))
    st.out = out
    return st


def _prepare_greedy(case, seed):
    st, dev = State(), _device()
    B, K, V = case["batch"], case["k"], case["vocab"]
    t = _logits(_gen(seed, 3), B * (K + 1), V)
    d = t.reshape(B, K + 1, V)[:, :K].argmax(2).to(torch.int32)
    # every sequence is refused at a place of its own
    for b in range(B):
        d[b, min(K - 1, b % (K + 1))] += 1 if b % (K + 1) < K else 0
    d = d.contiguous()
    tok = torch.empty(B, K + 1, dtype=torch.int32, device="cuda")
    acc = torch.empty(B, dtype=torch.int32, device="cuda")
    a = H.AcceptArgs(B, K, V, st.ptr(t), None, st.ptr(d), K, 1.0, 0, None, st.ptr(tok), st.ptr(acc), None)
    L, ref = H.lib(), C.byref(a)
    st.keep.append(a)
    st.call = lambda: H.check(L.opure_accept_greedy(dev.h, ref))
    st.out = dict(tokens=tok, accepted=acc)
    return st


PREPARE = dict(step=_prepare_step, prompt=_prepare_prompt, layer=_prepare_layer, attention=_prepare_attention,
               gemv=_prepare_gemv, reject=_prepare_reject, sample=_prepare_sample, greedy=_prepare_greedy)


def prepare(case, seed):
    st = PREPARE[case["kind"]](case, seed)
    torch.cuda.synchronize()
    return st


def run(state):
    if state.engine is not None:
        return state.engine.forward_logits(state.tokens, state.vocab)[0]
    if state.graph is not None:
        _device().graph_launch(state.graph)
    else:
        state.call()
    return state.out


# ---- what a pass cannot do without ----------------------------------------------


def _linear_bytes(out, inn, w):
    return {"f32": 4 * out * inn, "i8": out * inn + 2 * out, "i4": out * inn // 2 + 4 * out * (inn // 128)}[w]


def _layer_work(case, rows, ctx_tokens, row_positions):
    """One layer over `rows` rows: every weight once, the cached tokens once, the
    rows' residual read and written, their K/V written."""
    h, nh, nkv, hd, ff, w = (case[k] for k in ("hidden", "heads", "kv", "hd", "ffn", "w"))
    shapes = [((nh + 2 * nkv) * hd, h), (h, nh * hd), (2 * ff, h), (h, ff)]
    eb = 4 if case["a"] == "f32" else 2
    return dict(bytes=sum(_linear_bytes(o, i, w) for o, i in shapes) + 2 * nkv * hd * eb * (ctx_tokens + rows) + 8 * rows * h,
                flops=2 * rows * sum(o * i for o, i in shapes) + 4 * nh * hd * row_positions)


def _spread(case):
    lens = _contexts(case)
    rows = case["rows"]
    cached = lens[0] if case.get("mode") == "prompt" else sum(lens)
    return cached, sum(n + j + 1 for n in lens for j in range(rows))


def work(case):
    kind = case["kind"]
    if kind == "layer":
        cached, seen = _spread(case)
        return _layer_work(case, case["batch"] * case["rows"], cached, seen)
    if kind in ("step", "prompt"):
        if kind == "step":
            (cached, seen), rows, scored = _spread(case), case["batch"] * case["rows"], case["batch"] * case["rows"]
        else:
            n = rows = case["tokens"]
            cached, seen, scored = 0, n * (n + 1) // 2, 1
        one = _layer_work(case, rows, cached, seen)
        return dict(bytes=case["layers"] * one["bytes"] + _linear_bytes(case["vocab"], case["hidden"], case["w"]) +
                    4 * scored * case["vocab"],
                    flops=case["layers"] * one["flops"] + 2 * scored * case["vocab"] * case["hidden"])
    if kind == "attention":
        cached, seen = _spread(case)
        eb, rows = 4 if case["a"] == "f32" else 2, case["batch"] * case["rows"]
        return dict(bytes=2 * case["kv"] * case["hd"] * eb * (cached + rows) + 2 * rows * case["heads"] * case["hd"] * eb,
                    flops=4 * case["heads"] * case["hd"] * seen)
    if kind == "gemv":
        eb = 4 if case["a"] == "f32" else 2
        y = case["out"] // (2 if case["swiglu"] else 1)
        return dict(bytes=_linear_bytes(case["out"], case["inn"], case["w"]) + eb * case["rows"] * (case["inn"] + y),
                    flops=2 * case["rows"] * case["out"] * case["inn"])
    if kind == "reject":
        # of each sequence: the rows up to its first refusal (at least one pair), and the distribution written
        return dict(bytes=case["batch"] * case["vocab"] * 4 * 3, flops=20 * case["batch"] * case["vocab"] * 2)
    if kind == "sample":
        return dict(bytes=case["rows"] * case["vocab"] * 4, flops=20 * case["rows"] * case["vocab"])
    return dict(bytes=case["batch"] * (case["k"] + 1) * case["vocab"] * 4, flops=case["batch"] * (case["k"] + 1) * case["vocab"])


# ---- 64-bit results ---------------------------------------------------------------


def _rope64(x, pos):
    """Adjacent pairs (2p, 2p+1) of [rows][heads][hd] turned by pos * theta^(-2p/hd)."""
    hd = x.shape[2]
    f = pos.double()[:, None] * THETA ** (-torch.arange(0, hd, 2, device="cuda").double() / hd)
    c, s = f.cos()[:, None, :], f.sin()[:, None, :]
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack((a * c - b * s, a * s + b * c), 3).flatten(2)


def _attend64(q, k, v, pos, scale):
    """q [rows][heads][hd] at positions pos over k, v [tokens][kv][hd]."""
    R, nh, hd = q.shape
    nkv = k.shape[1]
    out = torch.empty_like(q)
    mask = torch.arange(k.shape[0], device="cuda")[None, :] > pos[:, None]
    for n in range(nkv):
        qs = q[:, n * (nh // nkv):(n + 1) * (nh // nkv)].reshape(-1, hd)
        s = (qs @ k[:, n].T * scale).reshape(R, nh // nkv, -1)
        p = s.masked_fill_(mask[:, None, :], -math.inf).softmax(2).reshape(qs.shape[0], -1)
        out[:, n * (nh // nkv):(n + 1) * (nh // nkv)] = (p @ v[:, n]).reshape(R, nh // nkv, hd)
    return out


def _planes64(pool, pages, hd):
    """K and V [tokens][kv][hd] of these pages of one layer's pool, in 64 bits."""
    t = pool[pages].double()
    nkv = t.shape[2]
    k = t[:, 0].reshape(len(pages), nkv, PAGE, hd).permute(0, 2, 1, 3).reshape(-1, nkv, hd)
    v = t[:, 1].reshape(len(pages), nkv, hd, PAGE).permute(0, 3, 1, 2).reshape(-1, nkv, hd)
    return k, v


def _norm64(x, gain):
    return x * (x.square().mean(1, keepdim=True) + 1e-5).rsqrt() * gain.double()


def _attention64(case, q, cache, pool):
    """Paged attention of every sequence's rows."""
    R, hd, out = case["rows"], case["hd"], torch.empty_like(q)
    for b, n in enumerate(cache["lens"]):
        pages = torch.from_numpy(cache["table"][b, :(n + R + PAGE - 1) // PAGE]).long().cuda()
        k, v = _planes64(pool, pages, hd)
        pos = n + torch.arange(R, device="cuda")
        out[b * R:(b + 1) * R] = _attend64(q[b * R:(b + 1) * R], k[:n + R], v[:n + R], pos, hd ** -0.5)
    return out


def _layer64(case, seed, layer, x, pos, attend):
    """One layer; attend(q, k, v) stores the rows' k, v and returns the attention."""
    W = _layer_weights(case, seed, layer)
    nh, nkv, hd = case["heads"], case["kv"], case["hd"]
    y = _norm64(x, W["attn_norm"]) @ _dense(W["qkv"]).T
    q, k, v = y.split((nh * hd, nkv * hd, nkv * hd), 1)
    n = x.shape[0]
    q, k = _rope64(q.reshape(n, nh, hd), pos), _rope64(k.reshape(n, nkv, hd), pos)
    x = x + attend(q, k, v.reshape(n, nkv, hd)).reshape(n, -1) @ _dense(W["o"]).T
    g, u = (_norm64(x, W["mlp_norm"]) @ _dense(W["gate_up"]).T).chunk(2, 1)
    return x + (torch.nn.functional.silu(g) * u) @ _dense(W["down"]).T


def _paged64(case, cache, layer, pos):
    """attend() of _layer64 over a paged cache; what it stores goes to cache["pool64"][layer] too."""
    hd, R = case["hd"], case["rows"]
    pool = cache["pool"][layer].double()
    cache.setdefault("pool64", {})[layer] = pool

    def attend(q, k, v):
        seq = torch.arange(q.shape[0], device="cuda") // R
        page = torch.from_numpy(cache["table"]).long().cuda()[seq, pos // PAGE]
        slot = pos % PAGE
        pool[:, 0].view(-1, case["kv"], PAGE, hd)[page, :, slot] = k
        pool[:, 1].view(-1, case["kv"], hd, PAGE)[page, :, :, slot] = v
        return _attention64(case, q, cache, pool)
    return attend


def _positions(case, cache):
    return torch.tensor([n + j for n in cache["lens"] for j in range(case["rows"])], device="cuda")


def _exact_layers(case, seed, x, layers):
    cache = _cache(case, seed, layers)
    pos = _positions(case, cache)
    for i in range(layers):
        x = _layer64(case, seed, i, x, pos, _paged64(case, cache, i, pos))
        cache["pool64"][i] = cache["pool64"][i][:cache["n_tail"]].clone()
    return x, torch.stack([cache["pool64"][i] for i in range(layers)])


def _philox(seed, c0, c1, c2):
    """Word 0 of Philox4x32-10 (Salmon et al. 2011) at counter (c0, c1, c2, 0)."""
    M, c, k0, k1 = 0xFFFFFFFF, [c0, c1, c2, 0], seed & 0xFFFFFFFF, (seed >> 32) & 0xFFFFFFFF
    for _ in range(10):
        p0, p1 = 0xD2511F53 * c[0], 0xCD9E8D57 * c[2]
        c = [(p1 >> 32) ^ c[1] ^ k0, p1 & M, (p0 >> 32) ^ c[3] ^ k1, p0 & M]
        k0, k1 = (k0 + 0x9E3779B9) & M, (k1 + 0xBB67AE85) & M
    return c[0]


def _exact_reject(case, seed):
    t, q, d = _reject_inputs(case, seed)
    B, K = case["batch"], case["k"]
    dist = torch.empty(B, case["vocab"], dtype=torch.float64, device="cuda")
    for b in range(B):
        p = (t[b].double() / case["temperature"]).softmax(1)
        r = (q[b].double() / case["temperature"]).softmax(1)
        n = 0
        while n < K and (_philox(int(seed), n, b, 1) >> 8) * 2.0 ** -24 * r[n, d[b, n]].item() < p[n, d[b, n]].item():
            n += 1
        w = (p[n] - r[n]).clamp(min=0) if n < K else p[K]
        dist[b] = w / w.sum()
    return dict(tokens=None, accepted=None, dist=dist)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("sample", "greedy"):
        return None                      # ids alone
    if kind == "reject":
        return _exact_reject(case, seed)
    if kind == "gemv":
        d, x = _gemv_inputs(case, seed)
        y = x.double() @ _dense(d).T
        if case["swiglu"]:
            g, u = y.chunk(2, 1)
            y = torch.nn.functional.silu(g) * u
        return y
    if kind == "attention":
        cache = _cache(case, seed, 1)
        n = case["batch"] * case["rows"]
        q = _randn(_gen(seed, 3), n, case["heads"] * case["hd"]).to(DTYPE[case["a"]]).double()
        return _attention64(case, q.reshape(n, case["heads"], case["hd"]), cache, cache["pool"][0]).reshape(n, -1)
    if kind == "layer":
        x, kv = _exact_layers(case, seed, _randn(_gen(seed, 3), case["batch"] * case["rows"], case["hidden"]).double(), 1)
        return dict(x=x, kv=kv)
    emb, gain = _head_weights(case, seed)
    emb = _dense(emb)
    if kind == "step":
        tok = torch.from_numpy(_tokens(case, seed)).long().cuda().reshape(-1)
        x, kv = _exact_layers(case, seed, emb[tok], case["layers"])
        return dict(logits=(_norm64(x, gain) @ emb.T).reshape(case["batch"], case["rows"], -1), tokens=None, accepted=None,
                    length=None, kv=kv)
    r = np.random.RandomState((int(seed) * 7 + 3) & 0x7FFFFFFF)
    tok = torch.from_numpy(r.randint(case["vocab"], size=case["tokens"])).cuda()
    pos = torch.arange(case["tokens"], device="cuda")
    x = emb[tok]
    for i in range(case["layers"]):
        x = _layer64(case, seed, i, x, pos, lambda q, k, v: _attend64(q, k, v, pos, case["hd"] ** -0.5))
    return (_norm64(x[-1:], gain) @ emb.T)[0].cpu().numpy()


def tolerance(case):
    """About four times the error against 64 bits that the entry points show.
    Ids and counts are exact."""
    kind = case["kind"]
    if kind in ("sample", "greedy"):
        return "exact"
    if kind == "reject":
        return {"rel": 1e-6, "differ": 0.0}
    if kind in ("step", "prompt"):
        return {"rel": {"f32": 1e-5, "f16": 6e-3, "bf16": 3e-2}[case["a"]], "differ": 0.0}
    if kind == "layer":
        return {"rel": {"f32": 2e-6, "f16": 1.5e-3, "bf16": 1.1e-2}[case["a"]]}
    return {"rel": {"f32": 2e-6, "f16": 1e-3, "bf16": 8e-3}[case["a"]]}
