"""GPU parity of the whole verify step (opure_verify_step) against the CPU oracle.

- logits within max_abs 1e-4 (fp32 path) or 2e-2 (fp16/bf16 paths);
- the K/V rows the step appends agree with the oracle's;
- the in-step acceptance equals the oracle's acceptance applied to the same
  GPU logits, bit for bit, and equals the oracle's own decision (the token
  seeds give every row a top-1/top-2 gap above twice the logit bar);
- a K+1-row step equals K+1 single-row steps bit for bit (so greedy
  speculative decoding reproduces greedy decoding exactly on the GPU);
- a captured hipGraph replays to the eager result;
- rollback restores the cache and length as the oracle does.
"""
import ctypes as C

import numpy as np
import pytest

import opure_hip as H
import oracle as O
import spec_loop
from gpu_util import VerifyRunner, device_kv, device_model, say, top2_gap

pytestmark = pytest.mark.gpu

FMTS = [(O.W_F32, O.A_F32, 1e-4), (O.W_I8PC, O.A_F16, 2e-2), (O.W_I4G128, O.A_F16, 2e-2),
        (O.W_I4G128, O.A_BF16, 2e-2)]
FMT_IDS = ["f32", "i8-f16", "i4-f16", "i4-bf16"]
# token seeds whose oracle logits have every row's top-1/top-2 gap above twice
# the logit bar, so the GPU's greedy decisions must equal the oracle's
# (found by searching seeds on the oracle alone)
TOKEN_SEED = {"f32": 3, "i8-f16": 3, "i4-f16": 11, "i4-bf16": 11}


@pytest.fixture(scope="module")
def dev():
    d = H.Dev(0)
    yield d
    d.close()


def small_model(wfmt, afmt, n_layers=2, seed=5, tied=True, vocab=1024, hidden=256, ffn=512, heads=(4, 2), hd=64,
                max_pos=1024, theta=10000.0, attn_scale=0.125):
    return O.HostModel(n_layers=n_layers, hidden=hidden, n_heads=heads[0], n_kv_heads=heads[1], head_dim=hd,
                       ffn=ffn, vocab=vocab, wfmt=wfmt, afmt=afmt, attn_scale=attn_scale, theta=theta,
                       max_pos=max_pos, tied=tied, seed=seed, norm_jitter=0.1)


def self_drafts(m, kv_o, pool0, tokens, seq_len, seq=0):
    """Sequence `seq` drafts its own greedy continuation: row j+1 := argmax of
    row j, built one row at a time because row j depends on rows <= j."""
    toks = np.array(tokens, np.int32).copy()
    for j in range(toks.shape[1] - 1):
        kv_o.pool[...] = pool0
        lg = O.verify_forward(m, kv_o, toks, np.asarray(seq_len, np.int32))
        toks[seq, j + 1] = int(np.argmax(lg[seq, j]))
    kv_o.pool[...] = pool0
    return toks


def random_cache(m, B, ctx_max, n_pages, seed):
    rng = np.random.default_rng(seed)
    mp = (ctx_max + 15) // 16
    kv = O.HostKV(m, n_pages=n_pages, batch=B, max_pages_per_seq=mp)
    kv.fill_random(rng, 1.0)
    perm = rng.permutation(n_pages)
    for b in range(B):
        kv.page_table[b] = perm[b * mp:(b + 1) * mp]
    return kv


@pytest.mark.parametrize("hidden", [192, 1088, 4096, 4160])
@pytest.mark.parametrize("afmt", [O.A_F16, O.A_BF16], ids=["f16", "bf16"])
def test_layer_norm_rows_same_bits(dev, hidden, afmt):
    """opure_verify_layer over more than 16 rows normalises its residual in one
    launch (hidden up to 4096, past that in two): from the embedding rows its
    first layer appends the K/V that the whole step (whose embedding leaves the
    tile sums) appends, bit for bit."""
    if afmt == O.A_BF16:
        hidden = (hidden + 127) // 128 * 128
    say("layer norm rows", hidden, afmt)
    wfmt = O.W_I8PC if afmt == O.A_F16 else O.W_I4G128
    m = small_model(wfmt, afmt, n_layers=1, hidden=hidden, ffn=256, vocab=64, tied=wfmt != O.W_I4G128)
    B, R = 7, 3
    kv = random_cache(m, B, 48, B * 3 + 2, seed=hidden)
    tokens = np.random.default_rng(hidden).integers(0, 64, (B, R)).astype(np.int32)
    ctx = np.array([0, 5, 13, 14, 15, 30, 40], np.int32)
    dm = device_model(dev, m)
    pools = []
    dkv = device_kv(dev, m, kv)
    run = VerifyRunner(dev, dm, dkv, B, R, max_ctx=48)
    run.step(tokens, ctx)
    pools.append(dkv.get_pool())
    dkv = device_kv(dev, m, kv)
    x, sl = dev.upload(O.verify_embed(m, tokens)), dev.upload(ctx)
    a = H.VerifyLayerArgs(C.pointer(dm.desc), C.pointer(dkv.desc), 0, B, R, int(sl), 48, int(x))
    H.check(H.lib().opure_verify_layer(dev.h, C.byref(a)))
    dev.sync()
    pools.append(dkv.get_pool())
    assert np.array_equal(pools[0], pools[1]) and not np.array_equal(pools[0], kv.pool)


def check_prompt_step(dev, m, rows, start):
    """One prompt step of `rows` tokens behind `start` cached positions: the
    appended K/V of every layer, the last row's logits and their argmax against
    the oracle's row by row, within the bars above (bf16: one storage ulp more
    on K/V, whose values reach past 4); without logits the same K/V."""
    import npref
    afmt = m.cfg["afmt"]
    cap = (start + rows + 16) // 16 * 16
    kv = random_cache(m, 1, cap, cap // 16 + 3, seed=rows)
    tokens = np.random.default_rng(rows).integers(0, m.cfg["vocab"], (1, rows)).astype(np.int32)
    dm = device_model(dev, m)
    kv_o = O.HostKV(m, n_pages=kv.n_pages, batch=1, max_pages_per_seq=kv.max_pages)
    kv_o.pool[...], kv_o.page_table[...] = kv.pool, kv.page_table
    O.set_threads(16)
    try:
        want = O.verify_forward(m, kv_o, tokens, np.array([start], np.int32))[0, -1]
    finally:
        O.set_threads(1)
    io = dev.upload(np.concatenate([tokens[0], np.array([start], np.int32)]))
    lb, ob = dev.alloc(m.cfg["vocab"] * 4), dev.alloc(4)
    pools = []
    for logits in (True, False):
        dkv = device_kv(dev, m, kv)
        a = H.PromptArgs(C.pointer(dm.desc), C.pointer(dkv.desc), int(io), int(io) + 4 * rows, rows, start + rows,
                         int(lb) if logits else None, int(ob) if logits else None)
        H.check(H.lib().opure_prompt_step(dev.h, C.byref(a)))
        dev.sync()
        pools.append(dkv.get_pool())
    got = dev.download(lb, np.float32, (m.cfg["vocab"],))
    say("max_abs logits", np.abs(got - want).max())
    assert np.abs(got - want).max() <= 2e-2
    assert dev.download(ob, np.int32, (1,))[0] == np.argmax(got)
    g, w = npref.act_to_f32(pools[0], afmt), npref.act_to_f32(kv_o.pool, afmt)
    assert (np.abs(g - w) <= 2e-2 + (2.0 ** -7 * np.abs(w) if afmt == O.A_BF16 else 0.0)).all()
    assert np.array_equal(pools[0], pools[1])


@pytest.mark.parametrize("rows,start", [(17, 0), (33, 100), (130, 37), (300, 37), (777, 0)])
@pytest.mark.parametrize("wfmt,afmt,hd", [(O.W_I8PC, O.A_F16, 64), (O.W_I4G128, O.A_F16, 128), (O.W_I4G128, O.A_BF16, 64)],
                         ids=["i8-f16-hd64", "i4-f16-hd128", "i4-bf16-hd64"])
def test_prompt_step_matches_oracle(dev, wfmt, afmt, hd, rows, start):
    """A prompt of one sequence behind `start` cached positions (a page's
    middle), up to a batch's rows and past them, with and without K splits:
    the appended K/V of both layers, the last row's logits and their argmax
    against the oracle's row by row, within the bars above (bf16: one storage
    ulp more on K/V, whose values reach past 4); without logits the same K/V."""
    say("prompt step", wfmt, afmt, hd, rows, start)
    m = small_model(wfmt, afmt, hd=hd, ffn=2048, attn_scale=hd ** -0.5, tied=wfmt != O.W_I4G128)
    check_prompt_step(dev, m, rows, start)


@pytest.mark.parametrize("rows,hidden,heads,ffn", [(1437, 256, (32, 8), 2048), (1437, 2816, (4, 2), 512),
                                                   (257, 256, (4, 2), 8192), (2048, 512, (16, 8), 512)], ids=lambda v: str(v))
@pytest.mark.parametrize("wfmt,afmt,hd", [(O.W_I8PC, O.A_F16, 64), (O.W_I4G128, O.A_F16, 64), (O.W_I4G128, O.A_BF16, 64)],
                         ids=["i8-f16", "i4-f16", "i4-bf16"])
def test_prompt_step_gemm_shapes_match_oracle(dev, wfmt, afmt, hd, rows, hidden, heads, ffn):
    """Sizes at which a GEMM of the prompt step has between one and two
    workgroups a CU (int8 halves its column groups): QKV and gate/up (288 and
    384 workgroups), the residual ones (264), gate/up at the fewest rows past a
    batch's (384); and the most rows of a step."""
    say("prompt step shapes", wfmt, afmt, rows, hidden, heads, ffn)
    m = small_model(wfmt, afmt, hd=hd, hidden=hidden, heads=heads, ffn=ffn, attn_scale=hd ** -0.5, max_pos=2048,
                    tied=wfmt != O.W_I4G128)
    check_prompt_step(dev, m, rows, 0)


@pytest.mark.parametrize("wfmt,afmt,hd,heads,rows,start", [
    (O.W_I8PC, O.A_F16, 64, (8, 2), 48, 2103), (O.W_I4G128, O.A_BF16, 64, (16, 4), 240, 1000),
    (O.W_I4G128, O.A_F16, 128, (16, 2), 96, 517)], ids=lambda v: str(v))
def test_prompt_step_behind_a_long_cache_same_bits(dev, wfmt, afmt, hd, heads, rows, start):
    """Few rows behind a long cache take the split attention of the verify step
    (k_attn_prompt would leave most of the chip idle while it walks the cache):
    up to 256 rows the prompt step appends, in every layer, the K/V bits of a
    verify step over the same rows in parts of 16."""
    say("prompt step, long cache", wfmt, afmt, hd, heads, rows, start)
    parts = rows // 16
    m = small_model(wfmt, afmt, n_layers=3, hd=hd, heads=heads, ffn=1024, max_pos=4096, attn_scale=hd ** -0.5, tied=True)
    cap = (start + rows + 16) // 16 * 16
    kv = random_cache(m, 1, cap, cap // 16 + 3, seed=rows)
    tokens = np.random.default_rng(rows).integers(0, m.cfg["vocab"], rows).astype(np.int32)
    dm = device_model(dev, m)
    one = device_kv(dev, m, kv)
    io = dev.upload(np.concatenate([tokens, start + 16 * np.arange(parts, dtype=np.int32)]))
    a = H.PromptArgs(C.pointer(dm.desc), C.pointer(one.desc), int(io), int(io) + 4 * rows, rows, start + rows, None, None)
    H.check(H.lib().opure_prompt_step(dev.h, C.byref(a)))
    dev.sync()
    wide = H.DeviceKV(dev, m.cfg, kv.n_pages, parts, kv.max_pages)
    wide.set_pool(kv.pool)
    wide.set_page_table(np.repeat(kv.page_table, parts, axis=0))
    v = H.VerifyArgs()
    v.model, v.kv, v.batch, v.rows, v.max_ctx = C.pointer(dm.desc), C.pointer(wide.desc), parts, 16, start + rows
    v.tokens, v.seq_len = int(io), int(io) + 4 * rows
    H.check(H.lib().opure_verify_step(dev.h, C.byref(v)))
    dev.sync()
    assert np.array_equal(one.get_pool(), wide.get_pool())


@pytest.mark.parametrize("wfmt,afmt,hd", [(O.W_I8PC, O.A_F16, 64), (O.W_I4G128, O.A_BF16, 64), (O.W_I4G128, O.A_F16, 128),
                                          (O.W_I4G128, O.A_BF16, 128)], ids=["i8-f16-64", "i4-bf16-64", "i4-f16-128", "i4-bf16-128"])
def test_prompt_step_row_blocks_agree(dev, wfmt, afmt, hd):
    """64 heads and 2,041 rows behind 2,050 cached positions take 128 query rows a
    workgroup (the last one ragged); the same rows in two steps take 64.  Tiles
    start at multiples of 64 from position 0 either way, so the rows of the
    second layer's K/V agree within the bars above (their GEMMs may sum in
    another order)."""
    import npref
    say("prompt step row blocks", wfmt, afmt, hd)
    rows, start, half = 2041, 2050, 1021
    m = small_model(wfmt, afmt, hd=hd, heads=(64, 8), hidden=256, ffn=512, attn_scale=hd ** -0.5, max_pos=4096, tied=True)
    cap = 4096
    kv = random_cache(m, 1, cap, cap // 16 + 3, seed=hd)
    tokens = np.random.default_rng(hd).integers(0, m.cfg["vocab"], rows).astype(np.int32)
    dm = device_model(dev, m)
    io = dev.upload(np.concatenate([tokens, np.array([start, start + half], np.int32)]))
    pools = []
    for parts in ([(0, rows)], [(0, half), (half, rows)]):
        dkv = device_kv(dev, m, kv)
        for i, (a0, a1) in enumerate(parts):
            a = H.PromptArgs(C.pointer(dm.desc), C.pointer(dkv.desc), int(io) + 4 * a0, int(io) + 4 * (rows + i), a1 - a0,
                             start + a1, None, None)
            H.check(H.lib().opure_prompt_step(dev.h, C.byref(a)))
        dev.sync()
        pools.append(npref.act_to_f32(dkv.get_pool(), afmt))
    g, w = pools
    assert np.isfinite(g).all() and not np.array_equal(g[1], npref.act_to_f32(kv.pool, afmt)[1])
    assert (np.abs(g - w) <= 2e-2 + (2.0 ** -7 * np.abs(w) if afmt == O.A_BF16 else 0.0)).all()


def test_prompt_step_refuses(dev):
    """Rows a verify step takes or too many, fp32, another head size, an
    argmax without logits."""
    m = small_model(O.W_I8PC, O.A_F16)
    kv = random_cache(m, 1, 4096, 257, seed=1)
    for mod, code in (({}, H.OK), ({"rows": 16}, H.E_CAPACITY), ({"rows": 2049}, H.E_CAPACITY), ({"logits": None}, H.E_INVALID),
                      ({"max_ctx": 31}, H.E_CAPACITY)):
        dm, dkv = device_model(dev, m), device_kv(dev, m, kv)
        io, lb = dev.upload(np.zeros(2050, np.int32)), dev.alloc(m.cfg["vocab"] * 4 + 4)
        v = {"rows": 32, "max_ctx": max(64, mod.get("rows", 0)), "logits": int(lb), **mod}
        a = H.PromptArgs(C.pointer(dm.desc), C.pointer(dkv.desc), int(io), int(io) + 4 * 2049, v["rows"], v["max_ctx"], v["logits"],
                         int(lb) + m.cfg["vocab"] * 4)
        assert H.lib().opure_prompt_step(dev.h, C.byref(a)) == code, mod
        dev.sync()
    for m in (small_model(O.W_F32, O.A_F32), small_model(O.W_I8PC, O.A_F16, hd=96)):
        kv = random_cache(m, 1, 64, 8, seed=1)
        dm, dkv = device_model(dev, m), device_kv(dev, m, kv)
        a = H.PromptArgs(C.pointer(dm.desc), C.pointer(dkv.desc), int(io), int(io) + 4 * 2049, 32, 64, None, None)
        assert H.lib().opure_prompt_step(dev.h, C.byref(a)) == H.E_UNSUPPORTED


@pytest.mark.parametrize("fmt", FMTS, ids=FMT_IDS)
def test_verify_step_matches_oracle(dev, fmt):
    wfmt, afmt, tol = fmt
    say("verify small", FMT_IDS[FMTS.index(fmt)])
    m = small_model(wfmt, afmt, tied=wfmt != O.W_I4G128)
    B, R = 2, 5
    kv = random_cache(m, B, 320, 48, seed=7)
    seq_len = np.array([251, 96], np.int32)
    rng = np.random.default_rng(TOKEN_SEED[FMT_IDS[FMTS.index(fmt)]])
    tokens = rng.integers(0, m.cfg["vocab"], size=(B, R)).astype(np.int32)
    dm, dkv = device_model(dev, m), device_kv(dev, m, kv)
    run = VerifyRunner(dev, dm, dkv, B, R, max_ctx=320)
    want_pool = kv.pool.copy()
    kv_o = O.HostKV(m, n_pages=kv.n_pages, batch=B, max_pages_per_seq=kv.max_pages)
    kv_o.pool[...] = kv.pool
    kv_o.page_table[...] = kv.page_table
    # sequence 0 drafts the oracle's own greedy continuation, so acceptance is exercised
    tokens = self_drafts(m, kv_o, want_pool, tokens, seq_len, seq=0)
    kv_o.pool[...] = want_pool
    want = O.verify_forward(m, kv_o, tokens, seq_len)
    run.step(tokens, seq_len, accept=H.ACCEPT_GREEDY)
    got = run.get_logits()
    err = np.abs(got - want).max()
    say("max_abs logits", err)
    assert err <= tol
    # appended K/V rows
    gpool = dkv.get_pool()
    if afmt == O.A_F32:
        assert np.abs(gpool - kv_o.pool).max() <= 1e-4
    else:
        import npref
        assert np.abs(npref.act_to_f32(gpool, afmt) - npref.act_to_f32(kv_o.pool, afmt)).max() <= 2e-2
    # acceptance inside the step == oracle acceptance on the same GPU logits (bit-exact)
    out, acc = run.get_accept()
    w_out, w_acc = O.accept_greedy(got, tokens[:, 1:])
    assert np.array_equal(out, w_out) and np.array_equal(acc, w_acc)
    # and == the oracle's own decision (every row's gap clears twice the bar)
    o_out, o_acc = O.accept_greedy(want, tokens[:, 1:])
    assert top2_gap(want).min() > 2 * tol
    assert np.array_equal(out, o_out) and np.array_equal(acc, o_acc)
    say("accepted", acc, "oracle", o_acc)
    assert acc[0] == R - 1


@pytest.mark.parametrize("fmt", FMTS[:2], ids=FMT_IDS[:2])
def test_rows_equal_single_row_steps(dev, fmt):
    wfmt, afmt, _ = fmt
    m = small_model(wfmt, afmt)
    kv = random_cache(m, 1, 256, 16, seed=9)
    dm = device_model(dev, m)
    dkv = device_kv(dev, m, kv)
    tokens = np.array([[11, 22, 33, 44, 55, 66]], np.int32)
    multi = VerifyRunner(dev, dm, dkv, 1, 6, 256)
    multi.step(tokens, [150])
    lm = multi.get_logits()
    dkv.set_pool(kv.pool)
    one = VerifyRunner(dev, dm, dkv, 1, 1, 256)
    for j in range(6):
        one.step(tokens[:, j:j + 1], [150 + j])
        assert np.array_equal(one.get_logits()[0, 0], lm[0, j]), j


@pytest.mark.parametrize("vocab", [1024, 32768], ids=["lm-head-k_gemv", "lm-head-wave-per-tile"])
def test_graph_replay_equals_eager(dev, vocab):
    """Replays of a captured greedy verify step equal the eager step, with
    eager work between them; at 2048 vocabulary tiles the LM head accepts in
    its own launch, each replay with the next launch count."""
    m = small_model(O.W_I8PC, O.A_F16, vocab=vocab)
    kv = random_cache(m, 2, 256, 32, seed=13)
    dm, dkv = device_model(dev, m), device_kv(dev, m, kv)
    run = VerifyRunner(dev, dm, dkv, 2, 4, 256)
    tokens = np.array([[1, 2, 3, 4], [5, 6, 7, 8]], np.int32)
    run.step(tokens, [100, 30], accept=H.ACCEPT_GREEDY)
    eager = run.get_logits()
    eager_acc = run.get_accept()
    a = run.args(accept=H.ACCEPT_GREEDY)
    dev.graph_begin()
    H.check(H.lib().opure_verify_step(dev.h, C.byref(a)))
    g = dev.graph_end()
    for i in range(4):
        dev.fill_u32(run.logits, 0x7FC00000, 2 * 4 * m.cfg["vocab"])   # eager work between replays
        dev.fill_u32(run.out_tokens, 0xFFFFFFFF, 2 * 4)
        dev.sync()
        dev.graph_launch(g)
        dev.sync()
        assert np.array_equal(run.get_logits(), eager), i
        o, acc = run.get_accept()
        assert np.array_equal(o, eager_acc[0]) and np.array_equal(acc, eager_acc[1])
    dev.graph_destroy(g)


def test_verify_with_rollback_matches_oracle(dev):
    m = small_model(O.W_I8PC, O.A_F16)
    B, R = 2, 6
    kv = random_cache(m, B, 512, 64, seed=17)
    seq_len = np.array([300, 120], np.int32)
    kv_o = O.HostKV(m, n_pages=kv.n_pages, batch=B, max_pages_per_seq=kv.max_pages)
    kv_o.pool[...] = kv.pool
    kv_o.page_table[...] = kv.page_table
    tokens = np.random.default_rng(2).integers(0, m.cfg["vocab"], size=(B, R)).astype(np.int32)
    dm, dkv = device_model(dev, m), device_kv(dev, m, kv)
    run = VerifyRunner(dev, dm, dkv, B, R, 512)
    run.step(tokens, seq_len, accept=H.ACCEPT_GREEDY, rollback=True, poison=True, poison_bits=0x7E00,
             free_pages=True)
    got = run.get_logits()
    out, acc = run.get_accept()
    O.verify_forward(m, kv_o, tokens, seq_len)
    w_out, w_acc = O.accept_greedy(got, tokens[:, 1:])
    assert np.array_equal(acc, w_acc)
    new_len, freed, nf = O.kv_rollback(kv_o, m, R - 1, seq_len, acc, poison_bits=0x7E00)
    assert np.array_equal(dev.download(run.new_len, np.int32, (B,)), new_len)
    assert np.array_equal(dev.download(run.n_freed, np.int32, (B,)), nf)
    assert np.array_equal(dkv.get_page_table(), kv_o.page_table)
    gpool = dkv.get_pool()
    # rolled-back slots carry the poison on both sides; kept slots agree within tolerance
    assert np.array_equal(gpool == 0x7E00, kv_o.pool == 0x7E00)
    import npref
    keep = kv_o.pool != 0x7E00
    diff = np.abs(npref.act_to_f32(gpool, O.A_F16) - npref.act_to_f32(kv_o.pool, O.A_F16))
    assert diff[keep].max() <= 2e-2


@pytest.mark.parametrize("shape", [(2, 6, (260, 97)), (1, 16, (300,))], ids=["2x6", "1x16"])
@pytest.mark.parametrize("fmt", [(O.W_I8PC, O.A_F16), (O.W_F32, O.A_F32), (O.W_I4G128, O.A_BF16)],
                         ids=["i8-f16", "f32", "i4-bf16"])
def test_greedy_acceptance_in_lm_head_same_as_separate(dev, fmt, shape):
    """A vocabulary of 2048 tiles puts the LM head on the wave-per-tile kernel,
    whose last workgroup then accepts greedily and rolls back inside the
    launch.  Tokens, accepted lengths, new lengths, freed pages, page table and
    poisoned pool equal the separate acceptance launch's
    (opure_debug_set_greedy_acceptance), on two steps in a row (the second
    with the next launch count), and the oracle's acceptance of the logits.
    Shapes: two sequences of 6 rows, sequence 0 drafting its own greedy
    continuation; one sequence of 16 rows (the most rows a step takes), whose
    drafts past the eighth are moved off that continuation, so at most 8 are
    accepted and the rollback poisons 7 or more positions."""
    B, R, ctx = shape
    say("greedy acceptance in the LM head", fmt, "batch", B, "rows", R)
    m = small_model(*fmt, vocab=32768)
    kv = random_cache(m, B, 512, 64, seed=21)
    seq_len = np.array(ctx, np.int32)
    kv_o = O.HostKV(m, n_pages=kv.n_pages, batch=B, max_pages_per_seq=kv.max_pages)
    kv_o.pool[...] = kv.pool
    kv_o.page_table[...] = kv.page_table
    tokens = np.random.default_rng(8).integers(0, m.cfg["vocab"], size=(B, R)).astype(np.int32)
    tokens = self_drafts(m, kv_o, kv.pool.copy(), tokens, seq_len, seq=0)
    if R > 9:
        tokens[0, 9:] = (tokens[0, 9:] + 1) % m.cfg["vocab"]
    dm = device_model(dev, m)
    poison = 0x7E00 if fmt[1] != O.A_F32 else 0x7FC00000
    res = {}
    lib = H.lib()
    try:
        for mode in (H.GREEDY_SEPARATE, H.GREEDY_IN_LM_HEAD):
            H.check(lib.opure_debug_set_greedy_acceptance(dev.h, mode))
            outs = []
            for rep in range(2):
                dkv = device_kv(dev, m, kv)
                run = VerifyRunner(dev, dm, dkv, B, R, 512)
                run.step(tokens, seq_len, accept=H.ACCEPT_GREEDY, rollback=True, poison=True, poison_bits=poison,
                         free_pages=True)
                out, acc = run.get_accept()
                outs.append((run.get_logits(), out, acc, dev.download(run.new_len, np.int32, (B,)),
                             dev.download(run.n_freed, np.int32, (B,)), dev.download(run.freed, np.int32, (B, 8)),
                             dkv.get_page_table(), dkv.get_pool()))
            res[mode] = outs
    finally:
        H.check(lib.opure_debug_set_greedy_acceptance(dev.h, H.GREEDY_IN_LM_HEAD))
    sep, fus = res[H.GREEDY_SEPARATE], res[H.GREEDY_IN_LM_HEAD]
    for rep in range(2):
        for k, (x, y) in enumerate(zip(sep[rep], fus[rep])):
            if k == 5:   # freed entries past n_freed are not written
                for b in range(B):
                    n = int(sep[rep][4][b])
                    assert np.array_equal(x[b, :n], y[b, :n]), (rep, b)
            else:   # bit for bit (the fp32 poison is a NaN)
                assert np.array_equal(np.ascontiguousarray(x).view(np.uint8), np.ascontiguousarray(y).view(np.uint8)), (rep, k)
    logits, out, acc = fus[0][0], fus[0][1], fus[0][2]
    w_out, w_acc = O.accept_greedy(logits, tokens[:, 1:])
    assert np.array_equal(out, w_out) and np.array_equal(acc, w_acc)
    if R > 9:
        assert acc[0] <= 8
    elif fmt[1] != O.A_BF16:    # bf16 activations may part from the oracle's own greedy drafts
        assert acc[0] == R - 1
    say("accepted", acc.tolist(), "freed", fus[0][4].tolist())


def _full_width(wfmt, afmt, shape, n_layers, vocab, seed, attn_scale):
    h, nh, nkv, hd, ff = shape
    return O.HostModel(n_layers=n_layers, hidden=h, n_heads=nh, n_kv_heads=nkv, head_dim=hd, ffn=ff, vocab=vocab,
                       wfmt=wfmt, afmt=afmt, attn_scale=attn_scale, theta=500000.0, max_pos=8192 + 64,
                       tied=wfmt == O.W_I8PC, seed=seed)


# attn_scale 1.0 is the reference's literal (unscaled) attention; 1/sqrt(hd) the
# Llama-3 value used for the Llama-shaped configurations.  The 8B-shape bf16
# case runs one layer: the depth at which the 2e-2 logit bar holds end to end
# for a bf16 model (tests/test_gpu_c4_depth.py holds all 32 layers to it one
# layer at a time).  Token seeds give every row a top-2 gap above twice the bar.
@pytest.mark.parametrize("cfg", [
    ("c3-1b-int8-2layers-unscaled", O.W_I8PC, O.A_F16, (2048, 32, 8, 64, 8192), 128256, 2048, 6, 1.0, 2, 7),
    ("c3-1b-int8-2layers", O.W_I8PC, O.A_F16, (2048, 32, 8, 64, 8192), 128256, 2048, 6, 0.125, 2, 1),
    ("c4-8b-int4-1layer", O.W_I4G128, O.A_BF16, (4096, 32, 8, 128, 14336), 16384, 8192, 8, 128 ** -0.5, 1, 2),
], ids=lambda c: c[0] if isinstance(c, tuple) else str(c))
def test_full_width(dev, cfg):
    name, wfmt, afmt, shape, vocab, ctx, R, scale, n_layers, token_seed = cfg
    say("full width", name)
    m = _full_width(wfmt, afmt, shape, n_layers, vocab, seed=101, attn_scale=scale)
    kv = random_cache(m, 1, ctx + R, (ctx + R + 15) // 16, seed=5)
    seq_len = np.array([ctx], np.int32)
    tokens = np.random.default_rng(token_seed).integers(0, vocab, size=(1, R)).astype(np.int32)
    dm, dkv = device_model(dev, m), device_kv(dev, m, kv)
    run = VerifyRunner(dev, dm, dkv, 1, R, ctx + R)
    O.set_threads(16)
    try:
        kv_o = O.HostKV(m, n_pages=kv.n_pages, batch=1, max_pages_per_seq=kv.max_pages)
        kv_o.pool[...] = kv.pool
        kv_o.page_table[...] = kv.page_table
        tokens = self_drafts(m, kv_o, kv.pool, tokens, seq_len)   # the oracle's greedy continuation
        want = O.verify_forward(m, kv_o, tokens, seq_len)
    finally:
        O.set_threads(1)
    dkv.set_pool(kv.pool)
    run.step(tokens, seq_len, accept=H.ACCEPT_GREEDY)
    got = run.get_logits()
    err = np.abs(got - want).max()
    gap = top2_gap(want).min()
    tol = 2e-2
    say(name, "max_abs", err, "min top2 gap", gap)
    assert err <= tol
    assert gap > 2 * tol
    out, acc = run.get_accept()
    w_out, w_acc = O.accept_greedy(got, tokens[:, 1:])
    assert np.array_equal(out, w_out) and np.array_equal(acc, w_acc)
    o_out, o_acc = O.accept_greedy(want, tokens[:, 1:])
    assert np.array_equal(out, o_out) and np.array_equal(acc, o_acc)
    assert acc[0] == R - 1


def test_c1_shape_speculative_equals_greedy(dev):
    """SmolLM-135M shape (hidden 576, 9/3 heads, hd 64, ffn 1536, vocab 49152),
    4 target layers and a 1-layer draft, fp32, K=4: the GPU's speculative output
    equals its greedy output bit for bit, and the oracle's greedy tokens."""
    shape = dict(hidden=576, n_heads=9, n_kv_heads=3, head_dim=64, ffn=1536, vocab=49152, wfmt=O.W_F32,
                 afmt=O.A_F32, attn_scale=1.0, theta=10000.0, max_pos=512, tied=True, norm_jitter=0.0)
    tgt = O.HostModel(n_layers=4, seed=71, **shape)
    drf = O.HostModel(n_layers=1, seed=72, **shape)
    prompt = list(np.random.default_rng(0).integers(0, 49152, 32))
    n_new, K = 24, 4
    dms = {"t": device_model(dev, tgt), "d": device_model(dev, drf)}
    kvs = {}
    runners = {}
    for key, hm in (("t", tgt), ("d", drf)):
        kvh = O.HostKV(hm, n_pages=8, batch=1, max_pages_per_seq=8)
        kvh.page_table[0] = np.arange(8)
        kvs[key] = device_kv(dev, hm, kvh)

    def runner(key, R):
        if (key, R) not in runners:
            runners[(key, R)] = VerifyRunner(dev, dms[key], kvs[key], 1, R, 128)
        return runners[(key, R)]

    def gpu_step(key, toks, ctx):
        R = toks.shape[1]
        out = []
        for s in range(0, R, 16):            # long prompts are fed 16 rows at a time
            r = runner(key, min(16, R - s))
            r.step(toks[:, s:s + 16], [ctx + s])
            out.append(r.get_logits())
        return np.concatenate(out, axis=1)

    def gpu_accept(toks, ctx):
        r = runner("t", toks.shape[1])
        r.step(toks, [ctx], accept=H.ACCEPT_GREEDY)
        o, a = r.get_accept()
        return o[0], int(a[0])

    greedy_gpu, _ = spec_loop.greedy(gpu_step, prompt, n_new)
    spec_gpu, hist = spec_loop.speculative(gpu_step, gpu_accept, prompt, n_new, K)
    say("gpu greedy", greedy_gpu[:8], "accepted per step", hist)
    assert spec_gpu == greedy_gpu

    okv = {k: O.HostKV(hm, n_pages=8, batch=1, max_pages_per_seq=8) for k, hm in (("t", tgt), ("d", drf))}
    for k in okv:
        okv[k].page_table[0] = np.arange(8)
    models = {"t": tgt, "d": drf}

    def orc_step(key, toks, ctx):
        return O.verify_forward(models[key], okv[key], toks, np.array([ctx], np.int32))

    O.set_threads(16)
    try:
        greedy_orc, gaps = spec_loop.greedy(orc_step, prompt, n_new)
    finally:
        O.set_threads(1)
    # the prompt and seeds give every oracle step a top-1/top-2 gap well above
    # the fp32 logit bar (measured 3.3e-3), so the ids must agree exactly
    say("oracle min gap", min(gaps))
    assert min(gaps) > 1e-4
    assert greedy_orc == greedy_gpu


@pytest.mark.parametrize("fmt", FMTS[1:], ids=FMT_IDS[1:])
def test_batched_verify_rejection_matches_oracle(dev, fmt):
    """A batch of sequences with ragged contexts, more than 16 rows in all
    (the thin-GEMM path): logits against the oracle, then rejection sampling
    at temperature 0.8 inside the step and the per-sequence rollback, equal
    bit for bit to the oracle's acceptance of the same GPU logits."""
    wfmt, afmt, tol = fmt
    m = small_model(wfmt, afmt, tied=wfmt != O.W_I4G128)
    B, R, V = 6, 7, m.cfg["vocab"]
    rng = np.random.default_rng(31)
    kv = random_cache(m, B, 400, 6 * 25 + 10, seed=9)
    seq_len = rng.integers(20, 390, size=B).astype(np.int32)
    tokens = rng.integers(0, V, size=(B, R)).astype(np.int32)
    say("batched verify", FMT_IDS[FMTS.index(fmt)], "seq_len", seq_len.tolist())
    dm, dkv = device_model(dev, m), device_kv(dev, m, kv)
    run = VerifyRunner(dev, dm, dkv, B, R, max_ctx=400)
    kv_o = O.HostKV(m, n_pages=kv.n_pages, batch=B, max_pages_per_seq=kv.max_pages)
    kv_o.pool[...] = kv.pool
    kv_o.page_table[...] = kv.page_table
    # drafts sampled from random draft logits at the same temperature
    q = (rng.standard_normal((B, R - 1, V)) * 2).astype(np.float32)
    pos = np.repeat(np.arange(R - 1)[None], B, 0).ravel()
    seqs = np.repeat(np.arange(B)[:, None], R - 1, 1).ravel()
    tokens[:, 1:] = O.sample_rows(q.reshape(-1, V), 0.8, 99, pos, seqs, 0).reshape(B, R - 1)
    kv_o.pool[...] = kv.pool
    want = O.verify_forward(m, kv_o, tokens, seq_len)
    # the first half of the batch drafts with q = the target's own scores, so
    # every draft is accepted there (u * q(x) < p(x) for any u < 1)
    run.step(tokens, seq_len)
    q[: B // 2] = run.get_logits()[: B // 2, : R - 1]
    dev.write(run.draft_logits, q)
    run.step(tokens, seq_len, accept=H.ACCEPT_REJECTION, rollback=True, temperature=0.8, seed=99)
    got = run.get_logits()
    err = np.abs(got - want).max()
    say("max_abs logits", err)
    assert err <= tol
    out, acc = run.get_accept()
    w_out, w_acc, _ = O.accept_rejection(got, q, tokens[:, 1:], 0.8, 99)
    assert np.array_equal(acc, w_acc) and np.array_equal(out, w_out)
    new_len = dev.download(run.new_len, np.int32, (B,))
    assert np.array_equal(new_len, seq_len + acc + 1)
    assert (acc[: B // 2] == R - 1).all()
    say("accepted", acc.tolist())


def test_batched_verify_greedy_matches_oracle(dev):
    """More than 16 rows with greedy acceptance (argmax over stored logits)."""
    m = small_model(O.W_I8PC, O.A_F16)
    B, R = 4, 6
    kv = random_cache(m, B, 320, 4 * 20 + 8, seed=12)
    seq_len = np.array([300, 17, 150, 64], np.int32)
    rng = np.random.default_rng(4)
    tokens = rng.integers(0, m.cfg["vocab"], size=(B, R)).astype(np.int32)
    dm, dkv = device_model(dev, m), device_kv(dev, m, kv)
    run = VerifyRunner(dev, dm, dkv, B, R, max_ctx=320)
    kv_o = O.HostKV(m, n_pages=kv.n_pages, batch=B, max_pages_per_seq=kv.max_pages)
    kv_o.pool[...] = kv.pool
    kv_o.page_table[...] = kv.page_table
    tokens = self_drafts(m, kv_o, kv.pool.copy(), tokens, seq_len, seq=2)
    kv_o.pool[...] = kv.pool
    want = O.verify_forward(m, kv_o, tokens, seq_len)
    run.step(tokens, seq_len, accept=H.ACCEPT_GREEDY, rollback=True)
    got = run.get_logits()
    assert np.abs(got - want).max() <= 2e-2
    out, acc = run.get_accept()
    w_out, w_acc = O.accept_greedy(got, tokens[:, 1:])
    assert np.array_equal(out, w_out) and np.array_equal(acc, w_acc)
    assert acc[2] == R - 1


def test_prefill_256_rows_on_one_page_table_row(dev):
    """A 300-token prompt written by one verify step of 16 parts x 16 rows
    that share the prompt's page-table row (part b at start + 16 b: its rows see
    every earlier part's K/V, appended by the same launch before attention), a
    second of 2 parts, then a 12-row step: the last 12 rows' logits agree with
    the oracle's one pass over all 300 rows (the wide parts run every GEMV as a
    thin GEMM)."""
    m = small_model(O.W_I8PC, O.A_F16, max_pos=512)
    V, P = m.cfg["vocab"], 300
    mp = (P + 15) // 16
    kv = O.HostKV(m, n_pages=mp + 8, batch=1, max_pages_per_seq=mp)
    rng = np.random.default_rng(41)
    kv.page_table[0] = rng.permutation(mp + 8)[:mp]
    prompt = rng.integers(0, V, size=P).astype(np.int32)
    want = O.verify_forward(m, kv, prompt[None, :], np.array([0], np.int32))[0, -12:]
    dm = device_model(dev, m)
    wide = H.DeviceKV(dev, m.cfg, mp + 8, 16, mp)
    wide.set_page_table(np.repeat(kv.page_table, 16, axis=0))
    toks = dev.alloc(256 * 4)
    sl = dev.alloc(16 * 4)
    for start, parts in ((0, 16), (256, 2)):
        dev.write(toks, prompt[start:start + 16 * parts])
        dev.write(sl, np.arange(parts, dtype=np.int32) * 16 + start)
        a = H.VerifyArgs()
        a.model = C.pointer(dm.desc)
        a.kv = C.pointer(wide.desc)
        a.batch, a.rows, a.max_ctx = parts, 16, mp * 16
        a.tokens, a.seq_len, a.logits = int(toks), int(sl), None
        H.check(H.lib().opure_verify_step(dev.h, C.byref(a)))
    dev.sync()
    one = H.DeviceKV.__new__(H.DeviceKV)
    one.__dict__.update(wide.__dict__)
    one.desc = H.KV(int(wide.pool), mp + 8, 16, int(wide.page_table), mp)   # row 0 of the same table
    one.batch = 1
    run = VerifyRunner(dev, dm, one, 1, 12, mp * 16)
    run.step(prompt[None, 288:], [288])
    err = np.abs(run.get_logits()[0] - want).max()
    say("prefill 256 rows: last 12 rows max_abs", err)
    assert err <= 2e-2
