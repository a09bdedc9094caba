"""Decode attention over the paged KV cache (gmoe_kv_*, gmoe_attention*) against the
oracle's attend_one / KVCacheState restatement (oracle/attention.py), within the layer
tolerance (rtol 1e-3, atol 1e-4): single sequences across page and chunk boundaries,
continuous batches of sequences at different lengths, prompts prefilled in one call,
sliding windows, the C5 head shape, refusals, page reuse, and the async form."""
from __future__ import annotations

import numpy as np
import pytest

import garuda_amd as G
from garuda_amd.attention import KvCache
from oracle.attention import KvOracle
from tests.test_gpu_dense import _hip
from tests.test_gpu_parity import ATOL, RTOL, bits, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    d = G.Device(0, slab_bytes=64 << 20)
    yield d
    d.close()


def check(got, want, what):
    err = np.abs(got - want)
    assert np.allclose(got, want, rtol=RTOL, atol=ATOL), f"{what}: max err {err.max()}"


def test_one_sequence_across_pages_and_chunks(dev):
    nh, nkv, hd = 8, 2, 64
    rng = np.random.default_rng(0)
    with KvCache(dev, 2, nh, nkv, hd, block_size=16, max_positions=600, max_seqs=2) as kv:
        o = KvOracle(2, nh, nkv, hd, max_positions=600)
        s = kv.open_seq()
        for step in range(530):  # crosses 16-position pages and 256-position chunks
            q, k, v = rng.normal(size=(1, nh * hd)), rng.normal(size=(1, nkv * hd)), rng.normal(size=(1, nkv * hd))
            got = kv.attention(1, [s], q, k, v)
            want = o.attention(1, [s], q, k, v)
            if step % 37 == 0 or step in (255, 256, 257, 511, 512, 529):
                say(f"one sequence, step {step}")
                check(got, want, f"step {step}")
        assert kv.seq_len(s, 1) == 530 and kv.seq_len(s, 0) == 0


def test_continuous_batch_prefill_and_window(dev):
    nh, nkv, hd = 8, 8, 32
    rng = np.random.default_rng(1)
    with KvCache(dev, 1, nh, nkv, hd, block_size=8, max_positions=400, sliding_window=100, max_seqs=4) as kv:
        o = KvOracle(1, nh, nkv, hd, max_positions=400, sliding_window=100)
        seqs = [kv.open_seq() for _ in range(3)]
        # prompts of different lengths, each prefilled in one call (entries in order)
        for s, plen in zip(seqs, (5, 130, 17)):
            ids = [s] * plen
            q, k, v = (rng.normal(size=(plen, w)) for w in (nh * hd, nkv * hd, nkv * hd))
            check(kv.attention(0, ids, q, k, v), o.attention(0, ids, q, k, v), f"prefill seq {s}")
        # decode steps over all three at once, then with one sequence twice per call
        for step in range(60):
            ids = seqs if step % 3 else seqs + [seqs[1]]
            n = len(ids)
            q, k, v = (rng.normal(size=(n, w)) for w in (nh * hd, nkv * hd, nkv * hd))
            check(kv.attention(0, ids, q, k, v), o.attention(0, ids, q, k, v), f"decode step {step}")
        for s in seqs:
            assert kv.seq_len(s) == o.seq_len(s)


@pytest.mark.parametrize("nh,nkv,hd", [(32, 2, 256), (16, 2, 96), (8, 1, 128)])
def test_wide_heads_and_groups(dev, nh, nkv, hd):
    # heads wider than 128 (the wide-head kernel), widths not a multiple of 16, and
    # groups whose (head, column) items exceed one pass of the workgroup
    rng = np.random.default_rng(hd)
    with KvCache(dev, 1, nh, nkv, hd, block_size=16, max_positions=300, max_seqs=2) as kv:
        o = KvOracle(1, nh, nkv, hd, max_positions=300)
        seqs = [kv.open_seq() for _ in range(2)]
        ids = [seqs[0]] * 150 + [seqs[1]] * 70  # prompts across chunks, one call
        q, k, v = (rng.normal(size=(len(ids), w)) for w in (nh * hd, nkv * hd, nkv * hd))
        say(f"wide heads nh={nh} nkv={nkv} hd={hd}: prefill")
        check(kv.attention(0, ids, q, k, v), o.attention(0, ids, q, k, v), "prefill")
        for step in range(3):
            q, k, v = (rng.normal(size=(2, w)) for w in (nh * hd, nkv * hd, nkv * hd))
            check(kv.attention(0, seqs, q, k, v), o.attention(0, seqs, q, k, v), f"decode {step}")


def test_c5_head_shape(dev):
    # 32 query heads on 8 kv heads of 128, eight sequences
    nh, nkv, hd = 32, 8, 128
    rng = np.random.default_rng(2)
    with KvCache(dev, 1, nh, nkv, hd, block_size=16, max_positions=2048, max_seqs=8) as kv:
        o = KvOracle(1, nh, nkv, hd, max_positions=2048)
        seqs = [kv.open_seq() for _ in range(8)]
        ids = [s for s in seqs for _ in range(40)]  # 40-token prompts, one call
        q, k, v = (rng.normal(size=(len(ids), w)) for w in (nh * hd, nkv * hd, nkv * hd))
        check(kv.attention(0, ids, q, k, v), o.attention(0, ids, q, k, v), "c5 prefill")
        for step in range(3):
            q, k, v = (rng.normal(size=(8, w)) for w in (nh * hd, nkv * hd, nkv * hd))
            check(kv.attention(0, seqs, q, k, v), o.attention(0, seqs, q, k, v), f"c5 decode {step}")


def test_refusals_and_page_reuse(dev):
    nh, nkv, hd = 4, 2, 16
    rng = np.random.default_rng(3)
    with KvCache(dev, 1, nh, nkv, hd, block_size=4, max_positions=10, max_seqs=2, max_pages=4) as kv:
        a = kv.open_seq()
        b = kv.open_seq()
        with pytest.raises(G.CacheError):
            kv.open_seq()  # both sequence slots taken
        mk = lambda n: (rng.normal(size=(n, nh * hd)), rng.normal(size=(n, nkv * hd)), rng.normal(size=(n, nkv * hd)))
        kv.attention(0, [a] * 10, *mk(10))  # 3 pages
        with pytest.raises(G.CacheError):
            kv.attention(0, [a], *mk(1))  # context window of 10 exhausted
        with pytest.raises(G.CacheError):
            kv.attention(0, [b] * 5, *mk(5))  # needs 2 pages, 1 free: refused, nothing changes
        assert kv.seq_len(b) == 0
        with pytest.raises(G.InferenceError):
            kv.attention(0, [7], *mk(1))
        kv.close_seq(a)  # its pages return to the pool
        o = KvOracle(1, nh, nkv, hd, max_positions=10)
        q, k, v = mk(8)
        check(kv.attention(0, [b] * 8, q, k, v), o.attention(0, [b] * 8, q, k, v), "reused pages")


def test_async_matches_sync(dev):
    import ctypes as C
    hip = _hip()
    nh, nkv, hd, n = 8, 2, 64, 4
    rng = np.random.default_rng(4)
    qs, ks, vs = [rng.normal(size=(n, w)).astype(np.float32) for w in (nh * hd, nkv * hd, nkv * hd)]
    with KvCache(dev, 1, nh, nkv, hd) as A, KvCache(dev, 1, nh, nkv, hd) as B:
        sa = [A.open_seq() for _ in range(n)]
        sb = [B.open_seq() for _ in range(n)]
        want = A.attention(0, sa, qs, ks, vs)
        bufs = [C.c_void_p() for _ in range(4)]
        for b, a in zip(bufs, (qs, ks, vs, want)):
            assert hip.hipMalloc(C.byref(b), a.nbytes) == 0
        st = C.c_void_p()
        assert hip.hipStreamCreate(C.byref(st)) == 0
        try:
            for b, a in zip(bufs[:3], (qs, ks, vs)):
                assert hip.hipMemcpy(b, a.ctypes.data, a.nbytes, 1) == 0
            B.attention_async(0, sb, bufs[0].value, bufs[1].value, bufs[2].value, bufs[3].value, st.value)
            assert hip.hipStreamSynchronize(st) == 0
            got = np.empty_like(want)
            assert hip.hipMemcpy(got.ctypes.data, bufs[3], got.nbytes, 2) == 0
            assert np.array_equal(bits(got), bits(want))
        finally:
            hip.hipStreamDestroy(st)
            for b in bufs:
                hip.hipFree(b)


@pytest.mark.parametrize("bad", ["nan", "inf"])
def test_nan_or_infinite_score_gives_uniform_weights(dev, bad):
    # simd::softmax falls back to uniform weights on a NaN or +inf score (simd/mod.rs:132-158)
    from tests.test_attention_oracle import nan_inf_case
    (nh, nkv, hd), steps = nan_inf_case(bad)
    with KvCache(dev, 1, nh, nkv, hd, block_size=4, max_positions=64, max_seqs=1) as kv:
        o = KvOracle(1, nh, nkv, hd, max_positions=64)
        s = kv.open_seq()
        for pos, (q, k, v) in enumerate(steps):
            say(f"{bad} score, position {pos}")
            got = kv.attention(0, [s], q[None], k[None], v[None])
            want = o.attention(0, [s], q[None], k[None], v[None])
            assert np.isfinite(got).all()
            check(got, want, f"{bad} position {pos}")


def _prompt_calls(kv, seqs, sizes, q, k, v, per=None):
    """The sequences' prompts, laid end to end in q, k and v: in one call, or in calls of `per` tokens."""
    ids = [s for s, n in zip(seqs, sizes) for _ in range(n)]
    if per is None:
        return kv.attention(0, ids, q, k, v)
    cut = [slice(p, min(p + per, len(ids))) for p in range(0, len(ids), per)]
    return np.concatenate([kv.attention(0, ids[c], q[c], k[c], v[c]) for c in cut])


@pytest.mark.parametrize("nh,nkv,hd,bs,window,sizes", [
    (4, 1, 128, 16, 0, (17,)), (4, 1, 128, 16, 0, (32,)), (4, 1, 128, 16, 0, (33, 65)),  # tile edges: 64 tokens of 4 heads
    (8, 8, 64, 16, 0, (127, 129)), (6, 2, 96, 8, 0, (64, 43)), (16, 1, 32, 4, 0, (21, 9)),  # group 1, 3, 16
    (32, 8, 128, 16, 0, (300, 1)), (8, 2, 32, 16, 50, (200, 40)), (8, 2, 64, 5, 1, (70,)),  # windows, odd pages
    (4, 4, 128, 16, 0, (600,)), (7, 1, 64, 16, 129, (400,)),
])
def test_prompt_tiles_equal_single_tokens(dev, nh, nkv, hd, bs, window, sizes):
    # A call of several consecutive tokens runs tiles of 256 (token, head) rows on MFMA; the
    # same prompt in calls of at most 16 tokens runs the single-token kernels. Both are f32
    # softmax-weighted means of the values, so they differ by the rounding of the scores
    # (hd products each) and of the sums over the span, relative to the largest value: a bound
    # on the worst case (what the tiles keep of f32 precision is the next test's matter).
    rng = np.random.default_rng(hd + nh + len(sizes))
    n = sum(sizes)
    q, k, v = (rng.normal(size=(n, w)).astype(np.float32) for w in (nh * hd, nkv * hd, nkv * hd))
    kw = dict(block_size=bs, max_positions=700, sliding_window=window, max_seqs=2)
    say(f"tiles nh={nh} nkv={nkv} hd={hd} bs={bs} window={window} sizes={sizes}")
    with KvCache(dev, 1, nh, nkv, hd, **kw) as A, KvCache(dev, 1, nh, nkv, hd, **kw) as B:
        got = _prompt_calls(A, [A.open_seq() for _ in sizes], sizes, q, k, v)
        want = _prompt_calls(B, [B.open_seq() for _ in sizes], sizes, q, k, v, per=16)
        # a second call on the cache the first one filled, its positions odd against the tiles
        q2, k2, v2 = (rng.normal(size=(35, w)).astype(np.float32) for w in (nh * hd, nkv * hd, nkv * hd))
        got2 = A.attention(0, [0] * 35, q2, k2, v2)
        want2 = _prompt_calls(B, [0], [35], q2, k2, v2, per=16)
    u = 2.0 ** -24
    for gq, gk, gv, x, y in ((q, k, v, got, want), (q2, np.concatenate([k, k2]), np.concatenate([v, v2]), got2, want2)):
        qa, ka = np.abs(gq.reshape(-1, nh, hd)), np.abs(gk.reshape(-1, nkv, hd))
        # |q.k| / sqrt(hd) <= |q| |k| / sqrt(hd), whatever the rotation; each score is hd + 2 roundings
        s = (np.linalg.norm(qa, axis=2).max() * np.linalg.norm(ka, axis=2).max()) / np.sqrt(hd)
        bound = 2 * (2 * (hd + 2) * s + 700 + 32) * u * np.abs(gv).max()
        err = np.abs(x - y).max()
        assert err <= bound, f"err {err} bound {bound}"
        assert np.sqrt(np.mean((x - y) ** 2)) <= 1e-6 * np.sqrt(np.mean(y ** 2)) + bound / 50


def _attention64(nh, nkv, hd, window, q, k, v):
    """One sequence's contexts in 64 bits, rope_theta 1 (every pair turned by its position)."""
    n = len(q)
    pos = np.arange(n)[:, None, None]
    c, s = np.cos(pos.astype(np.float64)), np.sin(pos.astype(np.float64))

    def rot(x, heads):
        a = x.astype(np.float64).reshape(n, heads, hd // 2, 2)
        return np.stack([a[..., 0] * c - a[..., 1] * s, a[..., 0] * s + a[..., 1] * c], -1).reshape(n, heads, hd)

    qr, kr, vv = rot(q, nh), rot(k, nkv), v.astype(np.float64).reshape(n, nkv, hd)
    i = np.arange(n)
    seen = (i[None] <= i[:, None]) & ((window == 0) | (i[None] > i[:, None] - window))
    out = np.empty((n, nh, hd))
    for h in range(nh):
        sc = np.where(seen, qr[:, h] @ kr[:, h * nkv // nh].T / np.sqrt(hd), -np.inf)
        w = np.exp(sc - sc.max(1, keepdims=True))
        out[:, h] = w @ vv[:, h * nkv // nh] / w.sum(1, keepdims=True)
    return out.reshape(n, nh * hd)


@pytest.mark.parametrize("nh,nkv,hd,n,window,qscale", [
    (4, 1, 128, 40, 0, 1.0), (8, 2, 128, 600, 0, 1.0), (8, 2, 128, 300, 70, 4.0), (8, 2, 32, 500, 0, 1.0),
    (4, 4, 64, 257, 0, 1.0), (6, 2, 96, 200, 0, 2.0)])
def test_prompt_tiles_are_as_precise_as_single_tokens(dev, nh, nkv, hd, n, window, qscale):
    # The tiles' products of three bf16 planes claim f32 precision: against the same attention
    # in 64 bits they must be no further off than the single-token kernels, whose products are
    # f32 (the maximum, one value of thousands, within twice theirs). Any of the six plane
    # products left out shows: the smallest of them are 2^-16 of a product, 250 f32 roundings.
    rng = np.random.default_rng(n + hd)
    q, k, v = (rng.normal(size=(n, w)).astype(np.float32) for w in (nh * hd, nkv * hd, nkv * hd))
    q *= np.float32(qscale)
    kw = dict(max_positions=700, sliding_window=window, max_seqs=1, rope_theta=1.0)
    say(f"tile precision nh={nh} nkv={nkv} hd={hd} n={n} window={window} q x {qscale}")
    with KvCache(dev, 1, nh, nkv, hd, **kw) as A, KvCache(dev, 1, nh, nkv, hd, **kw) as B:
        tiles = _prompt_calls(A, [A.open_seq()], [n], q, k, v)
        single = _prompt_calls(B, [B.open_seq()], [n], q, k, v, per=16)
    want = _attention64(nh, nkv, hd, window, q, k, v)
    et, es = np.abs(tiles - want), np.abs(single - want)
    say(f"  rms {np.sqrt((et ** 2).mean()):.2e} single {np.sqrt((es ** 2).mean()):.2e}, max {et.max():.2e} single {es.max():.2e}")
    assert np.sqrt((et ** 2).mean()) <= 1.05 * np.sqrt((es ** 2).mean())
    assert et.max() <= 2 * es.max()


def test_prompt_tiles_round_to_both_sides(dev):
    # values in [1, 2) make every product positive: planes cut off instead of rounded would make
    # each sum too small, by about 2^-24 of itself on average; rounded ones cancel
    nh, nkv, hd, n = 8, 2, 64, 512
    rng = np.random.default_rng(11)
    q, k = (rng.normal(size=(n, w)).astype(np.float32) for w in (nh * hd, nkv * hd))
    v = (1 + rng.random(size=(n, nkv * hd))).astype(np.float32)
    say("tile bias")
    with KvCache(dev, 1, nh, nkv, hd, max_positions=512, max_seqs=1, rope_theta=1.0) as A:
        got = _prompt_calls(A, [A.open_seq()], [n], q, k, v)
    want = _attention64(nh, nkv, hd, 0, q, k, v)
    bias = ((got - want) / want).mean()
    say(f"  mean relative error {bias:.2e}")
    assert abs(bias) <= 2.0 ** -27


@pytest.mark.parametrize("what", ["nan value", "inf value", "nan key", "inf key", "nan query"])
def test_prompt_tiles_with_non_finite_rows(dev, what):
    # A later token's non-finite key or value leaves the earlier tokens of its key tile as
    # they are; the tokens that attend to it see what the single-token kernels give them.
    nh, nkv, hd, n, at = 4, 2, 64, 90, 41
    rng = np.random.default_rng(7)
    q, k, v = (rng.normal(size=(n, w)).astype(np.float32) for w in (nh * hd, nkv * hd, nkv * hd))
    val = np.float32("nan" if "nan" in what else "inf")
    dict(value=v, key=k, query=q)[what.split()[1]][at, 3] = val
    say(f"tiles with a {what}")
    with KvCache(dev, 1, nh, nkv, hd, max_positions=128, max_seqs=1) as A, \
            KvCache(dev, 1, nh, nkv, hd, max_positions=128, max_seqs=1) as B:
        got = _prompt_calls(A, [A.open_seq()], [n], q, k, v)
        want = _prompt_calls(B, [B.open_seq()], [n], q, k, v, per=16)
    assert np.isfinite(want[:at]).all() and np.isfinite(got[:at]).all()
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    ok = np.isfinite(want)
    assert np.allclose(got[ok], want[ok], rtol=RTOL, atol=ATOL)


@pytest.mark.parametrize("nh,nkv,hd,bs,window", [(6, 2, 96, 8, 0), (8, 1, 128, 16, 90), (16, 1, 32, 4, 0)])
def test_prompt_tiles_with_non_finite_rows_over_a_long_span(dev, nh, nkv, hd, bs, window):
    # several chunks of positions a row, non-finite rows in the cache and in the call, -inf scores
    # beside finite ones, and every score -inf: as the single-token kernels
    rng = np.random.default_rng(hd)
    n = 300
    q, k, v = (rng.normal(size=(n, w)).astype(np.float32) for w in (nh * hd, nkv * hd, nkv * hd))
    k[60, 5] = np.inf     # scores of either sign
    v[150, 7] = np.nan
    q[200:210] = 0.0      # rows of equal scores: NaN where the infinite key is seen
    q[230, :] = np.inf
    kw = dict(block_size=bs, max_positions=400, sliding_window=window, max_seqs=1, rope_theta=1.0)
    say(f"tiles with non-finite rows hd={hd} window={window}")
    with KvCache(dev, 1, nh, nkv, hd, **kw) as A, KvCache(dev, 1, nh, nkv, hd, **kw) as B:
        got = _prompt_calls(A, [A.open_seq()], [n], q, k, v, per=100)
        want = _prompt_calls(B, [B.open_seq()], [n], q, k, v, per=16)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    ok = np.isfinite(want)
    assert ok.any() and np.allclose(got[ok], want[ok], rtol=RTOL, atol=ATOL)


@pytest.mark.parametrize("nh,nkv,hd,bs,window,order,tokens", [
    (32, 8, 128, 16, 0, "pssps", (40, 1)), (8, 8, 64, 16, 0, "sspss", (33, 2)),  # group 1: runs from 32 tokens tile
    (16, 1, 32, 4, 70, "spspspss", (20, 1)), (8, 2, 96, 5, 0, "ssssssssssssssssssssp", (90, 1)),
    (8, 2, 64, 16, 0, "pssss", (9, 3)),  # nine tokens of four rows fill an eighth of a tile, too few to tile beside others
    (8, 2, 64, 16, 0, "pspss", (9, 7)), (64, 64, 32, 16, 0, "pssss", (40, 1))])
def test_prompts_beside_decoding_sequences(dev, nh, nkv, hd, bs, window, order, tokens):
    # One call of prompts (p) and decoding sequences (s) at their own lengths: the prompts' rows in
    # tiles, the others in tiles too or, where those would have many keys, token by token (64 kv
    # heads). Each sequence by itself in calls of at most 16 tokens: within the layer tolerance, and
    # the same bits token by token.
    rng = np.random.default_rng(len(order) + hd)
    w = (nh * hd, nkv * hd, nkv * hd)
    kw = dict(block_size=bs, max_positions=400, sliding_window=window, max_seqs=len(order))
    say(f"mixed call hd={hd} {order}")
    with KvCache(dev, 1, nh, nkv, hd, **kw) as A, KvCache(dev, 1, nh, nkv, hd, **kw) as B:
        ids, runs, at = [], [], 0
        for s, c in enumerate(order):
            assert A.open_seq() == B.open_seq() == s
            past = int(rng.integers(1, 200))
            x = [rng.normal(size=(past, y)).astype(np.float32) for y in w]
            for kv in (A, B):
                _prompt_calls(kv, [s], [past], *x, per=16)
            m = tokens["ps".index(c)]
            ids += [s] * m
            runs.append((s, c, slice(at, at + m)))
            at += m
        for turn in range(2):
            q, k, v = (rng.normal(size=(at, y)).astype(np.float32) for y in w)
            got = A.attention(0, ids, q, k, v)
            for s, c, r in runs:
                want = _prompt_calls(B, [s], [r.stop - r.start], q[r], k[r], v[r], per=16)
                if c == "s" and nkv == 64:
                    assert np.array_equal(bits(got[r]), bits(want)), f"sequence {s}"
                check(got[r], want, f"sequence {s}")


def test_large_decode_batch_is_the_same_bits_as_small_ones(dev):
    # above 16 sequences the entries go through device memory; each sequence's rotation and
    # append still ride in the attention's own launch
    nh, nkv, hd, n = 8, 2, 64, 37
    rng = np.random.default_rng(3)
    with KvCache(dev, 1, nh, nkv, hd, max_seqs=n) as A, KvCache(dev, 1, nh, nkv, hd, max_seqs=n) as B:
        a, b = [A.open_seq() for _ in range(n)], [B.open_seq() for _ in range(n)]
        for step in range(70):
            m = n - step % 3
            q, k, v = (rng.normal(size=(m, w)).astype(np.float32) for w in (nh * hd, nkv * hd, nkv * hd))
            got = A.attention(0, a[:m], q, k, v)
            want = np.concatenate([B.attention(0, b[i:min(i + 16, m)], q[i:i + 16], k[i:i + 16], v[i:i + 16])
                                   for i in range(0, m, 16)])
            assert np.array_equal(bits(got), bits(want)), f"step {step}"


@pytest.mark.parametrize("nh,nkv,hd,bs,window,bad", [
    (8, 2, 32, 16, 0, None), (32, 8, 128, 16, 70, None), (2, 2, 4, 8, 0, None), (16, 1, 256, 16, 0, None),
    (8, 2, 96, 16, 64, None), (32, 8, 128, 16, 0, "nan"), (8, 2, 32, 5, 0, "inf")])
def test_decode_launch_with_rotation_is_the_same_bits(dev, nh, nkv, hd, bs, window, bad):
    # Calls of different sequences rotate and append in the attention's own launch; a call
    # with a sequence twice takes the separate launches. Both run the same operations, so
    # rows of sequences 0 and 1 agree bit for bit across pages and chunks of 64 positions.
    rng = np.random.default_rng(hd + bs)
    with KvCache(dev, 1, nh, nkv, hd, block_size=bs, max_positions=400, sliding_window=window, max_seqs=3) as A, \
            KvCache(dev, 1, nh, nkv, hd, block_size=bs, max_positions=400, sliding_window=window, max_seqs=3) as B:
        a = [A.open_seq() for _ in range(2)]
        b = [B.open_seq() for _ in range(3)]
        for step in range(134):
            q, k, v = (rng.normal(size=(4, w)).astype(np.float32) for w in (nh * hd, nkv * hd, nkv * hd))
            if bad and step in (20, 90):
                q[0, 3], k[1, 2] = np.float32(bad), -np.float32(bad)
            n = 1 if step == 0 else 2  # the second sequence runs one position behind
            got = A.attention(0, a[:n], q[:n], k[:n], v[:n])
            want = B.attention(0, b[:n] + [b[2]] * 2, *(np.concatenate([x[:n], x[2:]]) for x in (q, k, v)))[:n]
            if step % 16 == 0 or 60 <= step < 68 or step > 126:
                say(f"step {step}")
            same = (bits(got) == bits(want)) | (np.isnan(got) & np.isnan(want))
            assert same.all(), f"step {step}: {np.count_nonzero(~same)} differ"


def test_pinned_entries_survive_until_their_call_has_run(dev):
    # Calls above 16 tokens put their entries (24 bytes) and tiles into two pinned halves of 512 KiB,
    # 35 calls of 600 tokens each: 150 calls queued without a wait go round both twice, then one of
    # 22000 tokens needs a larger buffer while calls are queued, and more follow. A cache whose
    # stream is waited for after every call gives the same contexts.
    import ctypes as C
    hip = _hip()
    nh, nkv, hd, n, big = 2, 1, 32, 600, 22000
    rng = np.random.default_rng(8)
    x = [rng.normal(size=(big, w * hd)).astype(np.float32) for w in (nh, nkv, nkv)]
    calls = [(i % 3, n) for i in range(150)] + [(3, big)] + [(i % 3, n) for i in range(4)]
    bufs = []

    def device(nbytes, src=None):
        b = C.c_void_p()
        assert hip.hipMalloc(C.byref(b), nbytes) == 0
        bufs.append(b)
        if src is not None:
            assert hip.hipMemcpy(b, src.ctypes.data, nbytes, 1) == 0
        return b.value

    kw = dict(block_size=16, max_positions=32000, sliding_window=100, max_seqs=4)
    try:
        d = [device(t.nbytes, t) for t in x]
        out = []
        say("pinned ring")
        for wait in (False, True):
            with KvCache(dev, 1, nh, nkv, hd, **kw) as kv:
                ids = [kv.open_seq() for _ in range(4)]
                o = device(4 * nh * hd * sum(m for _, m in calls))
                at, res = 0, np.empty((sum(m for _, m in calls), nh * hd), np.float32)
                for i, (s, m) in enumerate(calls):
                    r = 0 if m == big else 7 * i  # other rows every call
                    q, k, v = (b + 4 * r * t.shape[1] for b, t in zip(d, x))
                    kv.attention_async(0, [ids[s]] * m, q, k, v, o + 4 * nh * hd * at, 0)
                    at += m
                    if wait:
                        assert hip.hipDeviceSynchronize() == 0
                assert hip.hipDeviceSynchronize() == 0
                assert hip.hipMemcpy(res.ctypes.data, o, res.nbytes, 2) == 0
                out.append(res)
        assert np.isfinite(out[0]).all() and np.array_equal(bits(out[0]), bits(out[1]))
    finally:
        for b in bufs:
            hip.hipFree(b)


def test_decode_context_over_its_query(dev):
    # the context may lie over the call's q, as when a caller reuses the buffer
    import ctypes as C
    hip = _hip()
    nh, nkv, hd, n = 8, 2, 64, 3
    rng = np.random.default_rng(5)
    qkv = [rng.normal(size=(n, w)).astype(np.float32) for w in (nh * hd, nkv * hd, nkv * hd)]
    with KvCache(dev, 1, nh, nkv, hd) as A, KvCache(dev, 1, nh, nkv, hd) as B:
        want = A.attention(0, [A.open_seq() for _ in range(n)], *qkv)
        bufs = [C.c_void_p() for _ in range(3)]
        for buf, x in zip(bufs, qkv):
            assert hip.hipMalloc(C.byref(buf), x.nbytes) == 0
            assert hip.hipMemcpy(buf, x.ctypes.data, x.nbytes, 1) == 0
        try:
            B.attention_async(0, [B.open_seq() for _ in range(n)], *(x.value for x in bufs), bufs[0].value, 0)
            assert hip.hipDeviceSynchronize() == 0
            got = np.empty_like(want)
            assert hip.hipMemcpy(got.ctypes.data, bufs[0], got.nbytes, 2) == 0
            assert np.array_equal(bits(got), bits(want))
        finally:
            for buf in bufs:
                hip.hipFree(buf)
