"""Timed workloads of the library, through its public entry points.

Each case is one call (or one short run of calls) that a serving program makes:

  * `moe`: a mixture-of-experts feed-forward call on device buffers (`MoeLayer.forward_async`),
    at the shapes this repository measures: the Mixtral shape (d 4096, f 14336, 8 experts
    top-2; Q4_K, or Q3_K gate/up with Q4_K down) and the fine-grained one (d 2048, f 768,
    128 experts top-8; Q6_K gate/up, Q8_0 down, router logits given);
  * `proj`: the attention projections of some layers, q|k|v stacked and o, or the output
    head (`DenseWeight.forward_async`);
  * `attn_decode`, `attn_prefill`: attention over the paged KV cache, one token of every
    sequence, or whole prompts in chunks (`KvCache.attention_async`);
  * `model`: a request through `DecodeModel`: prompts, then decode steps on given tokens,
    with the logits that a sampler reads.

Weights are drawn in the fields of their block format (codes, sub-block scales, block
scale) on the GPU, so that `exact` reads the same values without a decoder.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import garuda_amd as G
from garuda_amd import moe as M
from garuda_amd.attention import KvCache

SHAPES = {"mixtral": dict(d=4096, f=14336, ne=8, k=2), "fine": dict(d=2048, f=768, ne=128, k=8),
          "synthetic": dict(d=256, f=512, ne=8, k=2)}
HEADS = {"32x8x128": (32, 8, 128), "8x2x32": (8, 2, 32)}
BLOCK = {"q3_k": (256, 110), "q4_k": (256, 144), "q6_k": (256, 210), "q8_0": (32, 34), "f32": (1, 4)}
TYPE_ID = {"q3_k": G.Q3_K, "q4_k": G.Q4_K, "q6_k": G.Q6_K, "q8_0": G.Q8_0, "f32": G.F32}
STD = 0.02
CHUNK = 256        # prompt positions an attention call takes, as the model's prefill does
ROOM = 32768       # positions a decoding sequence may take before it is closed
PAGE = 16
MODELS = {  # layers, experts' and projections' types, heads, vocabulary
    "mixtral": dict(layers=2, gu="q3_k", dn="q4_k", proj="q4_k", head="q6_k", heads="32x8x128", vocab=32000,
                    math="packed", theta=1e6),
    "synthetic": dict(layers=4, gu="f32", dn="f32", proj="f32", head="f32", heads="8x2x32", vocab=512, math="f32",
                      theta=1e4)}


def listed():
    return [
        # the smallest whole call: the synthetic engine (4 layers of d 256, f32 weights), one
        # sequence stepped token by token; launches and their gaps
        dict(name="synthetic_decode", kind="model", preset="synthetic", seqs=1, prompt=16, steps=24),
        # one token of a Mixtral-shape layer: single-user decode, bound by the weights' bytes
        dict(name="moe_q4k_1", kind="moe", shape="mixtral", gu="q4_k", dn="q4_k", math="packed", tokens=1, skew=False),
        # a small decode batch: the headline
        dict(name="moe_q4k_8", kind="moe", shape="mixtral", gu="q4_k", dn="q4_k", math="packed", tokens=8, skew=False),
        # a larger decode batch of ragged size, a handful of tokens an expert
        dict(name="moe_q4k_29", kind="moe", shape="mixtral", gu="q4_k", dn="q4_k", math="packed", tokens=29, skew=False),
        # prefill with Zipf-skewed expert loads, in the arithmetic of mmapped checkpoints ...
        dict(name="moe_q4k_512", kind="moe", shape="mixtral", gu="q4_k", dn="q4_k", math="packed", tokens=512, skew=True),
        # ... and of checkpoints expanded to f32 (the reference's default)
        dict(name="moe_q4k_512_f32", kind="moe", shape="mixtral", gu="q4_k", dn="q4_k", math="f32", tokens=512, skew=True),
        # many small experts, about four tokens each
        dict(name="moe_fine_64", kind="moe", shape="fine", gu="q6_k", dn="q8_0", math="packed", tokens=64, skew=False),
        # the attention projections of eight layers at a decode batch ...
        dict(name="proj_8", kind="proj", what="attn", layers=8, math="packed", tokens=8),
        # ... and of two layers over a ragged prefill chunk
        dict(name="proj_250", kind="proj", what="attn", layers=2, math="packed", tokens=250),
        # attention of eight decoding sequences over a window of 2048, four layers
        dict(name="attn_decode_2048", kind="attn_decode", heads="32x8x128", layers=4, seqs=8, window=2048),
        # a 1500-token prompt through four layers' attention
        dict(name="attn_prefill_1500", kind="attn_prefill", heads="32x8x128", layers=4, tokens=1500),
        # requests through a Mixtral-shape model of two layers: prompts, then decode steps
        dict(name="mixtral_requests", kind="model", preset="mixtral", seqs=4, prompt=120, steps=12),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("moe", "moe", "moe", "proj", "proj", "attn_decode", "attn_prefill", "model"))
    if kind == "moe":
        shape, gu, dn = rng.choice((("mixtral", "q4_k", "q4_k"), ("mixtral", "q3_k", "q4_k"), ("fine", "q6_k", "q8_0")))
        n = _log_int(rng, 1, 512)
        return dict(kind=kind, shape=shape, gu=gu, dn=dn, math=rng.choice(("packed", "packed", "f32")), tokens=n,
                    skew=shape == "mixtral" and n >= 64)
    if kind == "proj":
        what = rng.choice(("attn", "attn", "head"))
        return dict(kind=kind, what=what, layers=1 if what == "head" else rng.randint(1, 4),
                    math=rng.choice(("packed", "packed", "f32")), tokens=_log_int(rng, 1, 64 if what == "head" else 256))
    if kind == "attn_decode":
        return dict(kind=kind, heads=rng.choice(("32x8x128", "32x8x128", "8x2x32")), layers=rng.randint(1, 4),
                    seqs=rng.randint(1, 16), window=_log_int(rng, 64, 4096))
    if kind == "attn_prefill":
        return dict(kind=kind, heads=rng.choice(("32x8x128", "32x8x128", "8x2x32")), layers=rng.randint(1, 4),
                    tokens=_log_int(rng, 16, 1500))
    preset = rng.choice(("synthetic", "mixtral"))
    if preset == "synthetic":
        return dict(kind=kind, preset=preset, seqs=rng.randint(1, 4), prompt=_log_int(rng, 4, 200),
                    steps=rng.randint(4, 24))
    return dict(kind=kind, preset=preset, seqs=rng.randint(1, 4), prompt=_log_int(rng, 8, 256), steps=rng.randint(2, 12))


# ---- weights, drawn in the fields of their block format ----

def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _gen(seed, *tag):
    h = int(seed) & 0xFFFFFFFF
    for t in tag:
        h = (h * 1000003 + int(t) + 12345) & 0xFFFFFFFFFFFF
    return torch.Generator(device=_dev()).manual_seed(h)


def _codes(gen, nblk, width, mean, std, lo, hi):
    q = torch.randn(nblk, width, generator=gen, device=_dev())
    return q.mul_(std).add_(mean).round_().clamp_(lo, hi).to(torch.int16 if lo < 0 else torch.uint8)


def _scale(gen, nblk, mean):
    """f16 block scales within 15 % of `mean`."""
    return (mean * (0.85 + 0.3 * torch.rand(nblk, generator=gen, device=_dev()))).half()


def _fields(qt, n, gen):
    """n values of N(0, STD^2) in the fields of block type qt."""
    e = BLOCK[qt][0]
    nb = n // e
    if qt == "f32":
        return dict(x=torch.randn(n, generator=gen, device=_dev()) * STD)
    if qt == "q8_0":
        return dict(q=_codes(gen, nb, 32, 0.0, 48.0, -127, 127), d=_scale(gen, nb, STD / 48.0))
    if qt == "q4_k":  # value = d * sc * q - dmin * m, m = sc and dmin = 7.5 d: codes centred
        d = _scale(gen, nb, STD / (3.4 * 52))
        sc = torch.randint(41, 64, (nb, 8), generator=gen, device=_dev(), dtype=torch.uint8)
        return dict(q=_codes(gen, nb, 256, 7.5, 3.4, 0, 15), sc=sc, d=d, dmin=(d.float() * 7.5).half())
    nsub, lim, std, top = (16, 4, 1.7, 31) if qt == "q3_k" else (16, 32, 13.0, 127)
    mag = torch.randint(top * 2 // 3, top + 1, (nb, nsub), generator=gen, device=_dev(), dtype=torch.int16)
    sign = 1 - 2 * torch.randint(0, 2, (nb, nsub), generator=gen, device=_dev(), dtype=torch.int16)
    return dict(q=_codes(gen, nb, 256, 0.0, std, -lim, lim - 1), sc=mag * sign,
                d=_scale(gen, nb, STD / (std * top * 5 / 6)))


def _pack(qt, F):
    """The packed bytes of drawn fields."""
    if qt == "f32":
        return F["x"].view(torch.uint8)
    q, nb = F["q"], F["q"].shape[0]
    d = F["d"].view(torch.uint8).view(nb, 2)
    if qt == "q8_0":
        return torch.cat([d, q.to(torch.int8).view(torch.uint8)], 1).reshape(-1)
    if qt == "q4_k":
        sc = F["sc"]
        lo = (sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6)  # scales and, equal to them, mins
        s12 = torch.cat([lo, lo, (sc[:, 4:] & 15) | ((sc[:, 4:] & 15) << 4)], 1)
        v = q.view(nb, 4, 2, 32)
        return torch.cat([d, F["dmin"].view(torch.uint8).view(nb, 2), s12, (v[:, :, 0] | (v[:, :, 1] << 4)).view(nb, 128)],
                         1).reshape(-1)
    if qt == "q6_k":
        v = (q + 32).to(torch.uint8).view(nb, 2, 4, 32)
        lo, hi = v & 15, v >> 4
        ql = torch.cat([lo[:, :, 0] | (lo[:, :, 2] << 4), lo[:, :, 1] | (lo[:, :, 3] << 4)], 2)
        qh = hi[:, :, 0] | (hi[:, :, 1] << 2) | (hi[:, :, 2] << 4) | (hi[:, :, 3] << 6)
        return torch.cat([ql.reshape(nb, 128), qh.reshape(nb, 64), F["sc"].to(torch.int8).view(torch.uint8), d], 1).reshape(-1)
    v = (q + 4).to(torch.uint8).view(nb, 2, 4, 32)  # q3_k: half, shift, byte
    q2, hb = v & 3, v >> 2
    qs = q2[:, :, 0] | (q2[:, :, 1] << 2) | (q2[:, :, 2] << 4) | (q2[:, :, 3] << 6)
    hm = torch.zeros(nb, 32, dtype=torch.uint8, device=q.device)
    for half in range(2):
        for j in range(4):
            hm |= hb[:, half, j] << (4 * half + j)
    s = (F["sc"] + 32).to(torch.uint8)
    top = s >> 4
    s8 = (s[:, :8] & 15) | ((s[:, 8:] & 15) << 4)
    s4 = top[:, :4] | (top[:, 4:8] << 2) | (top[:, 8:12] << 4) | (top[:, 12:] << 6)
    return torch.cat([hm, qs.reshape(nb, 64), s8, s4, d], 1).reshape(-1)


def _values(qt, F):
    """The f64 values of drawn fields."""
    if qt == "f32":
        return F["x"].double()
    nb = F["q"].shape[0]
    d, q = F["d"].double().view(nb, 1, 1), F["q"].double()
    if qt == "q8_0":
        return (d[:, 0] * q).reshape(-1)
    sc = F["sc"].double()
    ns = sc.shape[1]
    w = d * sc.view(nb, ns, 1) * q.view(nb, ns, 256 // ns)
    if qt == "q4_k":
        w -= F["dmin"].double().view(nb, 1, 1) * sc.view(nb, ns, 1)
    return w.reshape(-1)


def _bytes(qt, n):
    e, b = BLOCK[qt]
    return n // e * b


def _host(qt, parts, seed, *tag):
    """Host bytes of consecutive matrices of `parts` values each, every one drawn by itself."""
    out = np.empty(sum(_bytes(qt, n) for n in parts), np.uint8)
    at = 0
    for i, n in enumerate(parts):
        b = _pack(qt, _fields(qt, n, _gen(seed, *tag, i)))
        torch.from_numpy(out[at:at + b.numel()]).copy_(b)
        at += b.numel()
    return out


def _matrix(qt, rows, cols, seed, *tag):
    return _values(qt, _fields(qt, rows * cols, _gen(seed, *tag))).view(rows, cols)


def _normal(shape, seed, *tag):
    return torch.randn(*shape, generator=_gen(seed, *tag), device=_dev())


# ---- what a program holds before the call ----

class _State:
    """The objects of one prepared case; closed when the program drops it."""

    def __init__(self):
        self._owned = []

    def own(self, close):
        self._owned.append(close)

    def __del__(self):
        while self._owned:
            self._owned.pop()()


_side = None


def _stream():
    """The program's stream: every call of every state runs in its order."""
    global _side
    if _side is None:
        _side = torch.cuda.Stream()
    return _side.cuda_stream


def _router(case_shape, seed, skew, layer=0):
    s = SHAPES[case_shape]
    r = (_normal((s["ne"], s["d"]), seed, 40, layer) * STD).cpu().numpy()
    if skew:
        r = M.skew_router(r, s["ne"], s["d"], M.skew_direction(seed & 0xFFFF, s["d"])).reshape(s["ne"], s["d"])
    return np.ascontiguousarray(r, np.float32)


def _tokens_in(case, seed):
    s = SHAPES[case["shape"]]
    hs = _normal((case["tokens"], s["d"]), seed, 50)
    if case["skew"]:
        hs = torch.from_numpy(M.skew_tokens(hs.cpu().numpy(), M.skew_direction(seed & 0xFFFF, s["d"]))).to(_dev())
    return hs


def _logits_in(case, seed):
    if case["shape"] != "fine":
        return None
    return 4.0 * torch.rand(case["tokens"], SHAPES["fine"]["ne"], generator=_gen(seed, 60), device=_dev())


def _experts(shape, gu, dn, seed, layer=0):
    s = SHAPES[shape]
    return [_host(qt, [s["d"] * s["f"]] * s["ne"], seed, 10 + p, layer) for p, qt in enumerate((gu, gu, dn))]


def _slab(shape, gu, dn, layers=1):
    s = SHAPES[shape]
    n = s["d"] * s["f"]
    return layers * s["ne"] * (int(1.08 * (2 * _bytes(gu, n) + _bytes(dn, n))) + 4096) + (64 << 20)


def _math(name):
    return G.MATH_PACKED if name == "packed" else G.MATH_F32


def _device(st, slab_bytes):
    dev = G.Device(0, slab_bytes=slab_bytes)
    st.own(dev.close)
    return dev


def _layer(st, dev, shape, gu, dn, seed, math_, skew=False, layer=0, **kw):
    s = SHAPES[shape]
    m = G.MoeLayer(dev, s["d"], s["f"], s["ne"], s["k"], _router(shape, seed, skew, layer),
                   *_experts(shape, gu, dn, seed, layer), tuple(TYPE_ID[t] for t in (gu, gu, dn)), math=_math(math_), **kw)
    st.own(m.release)
    return m


def _dense(st, dev, qt, rows, cols, math_, seed, *tag):
    w = G.DenseWeight(dev, TYPE_ID[qt], rows, cols, _host(qt, [rows * cols], seed, *tag), _math(math_))
    st.own(w.release)
    return w


def _proj_shapes(case):
    if case["what"] == "head":
        return (("q6_k", 32000, 4096),)
    return (("q4_k", 6144, 4096), ("q4_k", 4096, 4096))  # q|k|v, o


def _prepare_moe(case, seed, st):
    s, n = SHAPES[case["shape"]], case["tokens"]
    st.dev = _device(st, _slab(case["shape"], case["gu"], case["dn"]))
    st.layer = _layer(st, st.dev, case["shape"], case["gu"], case["dn"], seed, case["math"], case["skew"])
    st.n, st.hs, st.logits = n, _tokens_in(case, seed), _logits_in(case, seed)
    st.out = torch.empty(n, s["d"], device="cuda")
    st.ids = torch.empty(n, s["k"], dtype=torch.int32, device="cuda")
    st.w = torch.empty(n, s["k"], device="cuda")


def _run_moe(st):
    st.layer.forward_async(st.hs.data_ptr(), st.n, st.out.data_ptr(), st.ids.data_ptr(), st.w.data_ptr(),
                           st.logits.data_ptr() if st.logits is not None else 0, _stream())
    return dict(out=st.out, ids=st.ids, weights=st.w)


def _prepare_proj(case, seed, st):
    n = st.n = case["tokens"]
    st.dev = _device(st, 1 << 20)
    st.calls = []
    for l in range(case["layers"]):
        for j, (qt, rows, cols) in enumerate(_proj_shapes(case)):
            w = _dense(st, st.dev, qt, rows, cols, case["math"], seed, 20 + j, l, 0)
            st.calls.append((w, _normal((n, cols), seed, 30 + j, l), torch.empty(n, rows, device="cuda")))


def _run_proj(st):
    for w, x, out in st.calls:
        w.forward_async(x.data_ptr(), st.n, out.data_ptr(), _stream())
    return [out for _, _, out in st.calls]


def _attn_inputs(heads, layers, n, seed, tag):
    nh, nkv, hd = HEADS[heads]
    return [tuple(_normal((n, w * hd), seed, tag, l, i) for i, w in enumerate((nh, nkv, nkv))) for l in range(layers)]


def _attend(kv, layer, seqs, qkv, out, at=0):
    q, k, v = qkv
    kv.attention_async(layer, seqs, *(t.data_ptr() + at * t.shape[1] * 4 for t in (q, k, v)),
                       out.data_ptr() + at * out.shape[1] * 4, _stream())


def _prepare_attn_decode(case, seed, st):
    nh, nkv, hd = HEADS[case["heads"]]
    n, nl, win = case["seqs"], case["layers"], case["window"]
    st.dev, st.layers, st.room = _device(st, 1 << 20), nl, ROOM - win
    st.kv = KvCache(st.dev, nl, nh, nkv, hd, block_size=PAGE, max_positions=ROOM, sliding_window=win, max_seqs=n)
    st.own(st.kv.close)
    st.qkv = _attn_inputs(case["heads"], nl, n, seed, 70)
    st.past = [_normal((n, win, 2 * nkv * hd), seed, 71, l) for l in range(nl)]
    st.out = [torch.empty(n, nh * hd, device="cuda") for _ in range(nl)]
    st.n, st.win, st.kvd, st.qd = n, win, nkv * hd, nh * hd
    _fill(st)


def _fill(st):
    """The sequences' first `window` positions in every layer."""
    st.seqs = [st.kv.open_seq() for _ in range(st.n)]
    st.done = 0
    torch.cuda.synchronize()
    for p in range(0, st.win, 64):
        m = min(64, st.win - p)
        seqs = [s for s in st.seqs for _ in range(m)]
        q, out = torch.zeros(st.n * m, st.qd, device="cuda"), torch.empty(st.n * m, st.qd, device="cuda")
        for l in range(st.layers):
            past = st.past[l][:, p:p + m].reshape(st.n * m, -1)
            k, v = past[:, :st.kvd].contiguous(), past[:, st.kvd:].contiguous()
            torch.cuda.synchronize()
            _attend(st.kv, l, seqs, (q, k, v), out)
            torch.cuda.synchronize()


def _run_attn_decode(st):
    if st.done == st.room:  # the window's room is used up: the sequences start again
        for s in st.seqs:
            st.kv.close_seq(s)
        _fill(st)
    st.done += 1
    for l in range(st.layers):
        _attend(st.kv, l, st.seqs, st.qkv[l], st.out[l])
    return st.out


def _prepare_attn_prefill(case, seed, st):
    nh, nkv, hd = HEADS[case["heads"]]
    st.n, st.layers = case["tokens"], case["layers"]
    st.dev = _device(st, 1 << 20)
    st.kv = KvCache(st.dev, st.layers, nh, nkv, hd, block_size=PAGE, max_positions=2048, max_seqs=1)
    st.own(st.kv.close)
    st.qkv = _attn_inputs(case["heads"], st.layers, st.n, seed, 70)
    st.out = [torch.empty(st.n, nh * hd, device="cuda") for _ in range(st.layers)]


def _run_attn_prefill(st):
    s = st.kv.open_seq()
    for p in range(0, st.n, CHUNK):
        m = min(CHUNK, st.n - p)
        for l in range(st.layers):
            _attend(st.kv, l, [s] * m, st.qkv[l], st.out[l], p)
    st.kv.close_seq(s)
    return st.out


def _norm_weight(d, seed, i):
    return 1.0 + 0.05 * _normal((d,), seed, 80, i)


def _prompt(case, seed):
    vocab = MODELS[case["preset"]]["vocab"]
    g = torch.Generator().manual_seed(int(seed) & 0xFFFFFFFF)
    return torch.randint(0, vocab, (case["seqs"], case["prompt"] + case["steps"]), generator=g).numpy().astype(np.uint32)


def _prepare_model(case, seed, st):
    c, s = MODELS[case["preset"]], SHAPES[case["preset"]]
    nh, nkv, hd = HEADS[c["heads"]]
    d, nl = s["d"], c["layers"]
    dev = st.dev = _device(st, _slab(case["preset"], c["gu"], c["dn"], nl))
    kw = dict(gating=G.GATING_MIXTRAL, combine=G.COMBINE_RANK_ORDER) if case["preset"] == "synthetic" else {}
    layers = [_layer(st, dev, case["preset"], c["gu"], c["dn"], seed, c["math"], layer=l, **kw) for l in range(nl)]
    dense = [[_dense(st, dev, c["proj"], rows, cols, c["math"], seed, 20 + j, l, 0) for l in range(nl)]
             for j, (rows, cols) in enumerate(((nh * hd, d), (nkv * hd, d), (nkv * hd, d), (d, nh * hd)))]
    head = _dense(st, dev, c["head"], c["vocab"], d, c["math"], seed, 90)
    table = _host(c["head"], [c["vocab"] * d], seed, 91)
    st.kv = KvCache(dev, nl, nh, nkv, hd, block_size=PAGE, max_positions=2048, max_seqs=case["seqs"], rope_theta=c["theta"])
    norms = [_norm_weight(d, seed, i).cpu().numpy() for i in range(2 * nl + 1)]
    st.model = G.DecodeModel(dev, st.kv, layers, *dense, head, np.stack(norms[:nl]), np.stack(norms[nl:2 * nl]), norms[-1],
                             (TYPE_ID[c["head"]], table, c["vocab"], d))
    st.own(st.kv.close)
    st.own(st.model.close)
    st.toks, st.prompt, st.by_step = _prompt(case, seed), case["prompt"], case["preset"] == "synthetic"


def _run_model(st):
    seqs = [st.kv.open_seq() for _ in st.toks]
    if st.by_step:  # the synthetic engine steps through its prompt
        for p in range(st.prompt - 1):
            st.model.decode_step(seqs, st.toks[:, p])
        first = st.model.decode_step(seqs, st.toks[:, st.prompt - 1], want_logits=True)[1]
    else:
        first = np.concatenate([st.model.prefill(s, t[:st.prompt], want_logits=True)[1] for s, t in zip(seqs, st.toks)])
    logits = [first]
    for p in range(st.prompt, st.toks.shape[1]):
        logits.append(st.model.decode_step(seqs, st.toks[:, p], want_logits=True)[1])
    for s in seqs:
        st.kv.close_seq(s)
    return np.stack(logits)


_KINDS = {"moe": (_prepare_moe, _run_moe), "proj": (_prepare_proj, _run_proj),
          "attn_decode": (_prepare_attn_decode, _run_attn_decode),
          "attn_prefill": (_prepare_attn_prefill, _run_attn_prefill), "model": (_prepare_model, _run_model)}


def prepare(case, seed):
    st = _State()
    st.run = _KINDS[case["kind"]][1]
    _KINDS[case["kind"]][0](case, seed, st)
    torch.cuda.synchronize()
    return st


def run(st):
    return st.run(st)


# ---- what a pass cannot do without ----

def _moe_work(s, gu, dn, n, router=True):
    touched = s["ne"] * (1.0 - (1.0 - s["k"] / s["ne"]) ** n)
    m = s["d"] * s["f"]
    return (touched * (2 * _bytes(gu, m) + _bytes(dn, m)) + s["ne"] * s["d"] * 4 * router + 2 * n * s["d"] * 4,
            6.0 * n * s["k"] * m)


def _attn_work(heads, n_in, kv_read, pairs):
    nh, nkv, hd = HEADS[heads]
    return 4.0 * (2 * n_in * nh * hd + 4 * n_in * nkv * hd + 2 * kv_read * nkv * hd), 4.0 * pairs * nh * hd


def work(case):
    kind = case["kind"]
    if kind == "moe":
        s = SHAPES[case["shape"]]
        b, f = _moe_work(s, case["gu"], case["dn"], case["tokens"], case["shape"] != "fine")
        b += case["tokens"] * (s["k"] * 8 + (s["ne"] * 4 if case["shape"] == "fine" else 0))
    elif kind == "proj":
        n = case["tokens"]
        b = case["layers"] * sum(_bytes(qt, r * c) + 4.0 * n * (r + c) for qt, r, c in _proj_shapes(case))
        f = case["layers"] * sum(2.0 * n * r * c for _, r, c in _proj_shapes(case))
    elif kind == "attn_decode":
        n = case["seqs"]
        b, f = (case["layers"] * v for v in _attn_work(case["heads"], n, n * case["window"], n * case["window"]))
    elif kind == "attn_prefill":
        n = case["tokens"]
        b, f = (case["layers"] * v for v in _attn_work(case["heads"], n, 0, n * (n + 1) // 2))
    else:
        c, s = MODELS[case["preset"]], SHAPES[case["preset"]]
        nh, nkv, hd = HEADS[c["heads"]]
        n, p, t, d = case["seqs"], case["prompt"], case["steps"], s["d"]
        # calls over the weights, tokens of each: the prompts (one each, or step by step), the steps
        calls = [(p, n)] * 1 if case["preset"] == "synthetic" else [(n, p)]
        calls.append((t, n))
        proj = d * (2 * nh + 2 * nkv) * hd
        b = f = 0.0
        for count, m in calls:
            mb, mf = _moe_work(s, c["gu"], c["dn"], m)
            b += count * c["layers"] * (mb + _bytes(c["proj"], proj))
            f += count * c["layers"] * (mf + 2.0 * m * proj)
        heads = (t + n if case["preset"] == "mixtral" else t + 1)  # calls of the output head
        b += heads * _bytes(c["head"], c["vocab"] * d) + 4.0 * n * (t + 1) * c["vocab"]
        f += 2.0 * n * (t + 1) * c["vocab"] * d
        reads = n * sum(range(p, p + t)) if case["preset"] == "mixtral" else n * sum(range(p + t))
        ab, af = _attn_work(c["heads"], n * (p + t), reads, n * (p + t) * (p + t + 1) // 2)
        b, f = b + c["layers"] * ab, f + c["layers"] * af
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    # Against `exact` the path showed (2-norm, relative): packed layers 5e-5 to 2e-4 (h is rounded to
    # int8 inside the layer, and a last-bit difference before that moves a code now and then), f32
    # layers 1.6e-6, projections and attention 1e-7 to 3e-7, which sums in another order may take
    # several times further, the f32 model 3e-7 and the packed model 1.2e-2 to 1.8e-2 (a code moved in
    # one layer travels through the next). Each bound is about four times that, or for f32 sums what a
    # plain order of them gives.
    if case["kind"] == "moe":
        return {"rel": 1e-3} if case["math"] == "packed" else {"rel": 8e-6}
    if case["kind"] in ("proj", "attn_decode", "attn_prefill"):
        return {"rel": 4e-6}
    return {"rel": 3e-2} if MODELS[case["preset"]]["math"] == "packed" else {"rel": 1e-5}


# ---- the same in 64 bits ----

def _int8(x):
    """Packed math's activations: int8 codes per 32 values, their scale max / 127 (quant/mod.rs:331-345)."""
    b = x.float().reshape(-1, 32)
    s = b.abs().amax(1, keepdim=True) / 127.0
    inv = torch.where(s > 0, 1.0 / s, torch.zeros_like(s))
    v = b * inv
    q = torch.where(v < 0, -torch.floor(-v + 0.5), torch.floor(v + 0.5)).clamp(-127, 127)  # halves away from 0
    return (s.double() * q.double()).reshape(x.shape)


def _mul(x, w, math_):
    return (_int8(x) if math_ == "packed" else x) @ w.t()


def _exact_moe(shape, gu, dn, math_, hs, router, logits, seed, layer=0, rank_softmax=False):
    s = SHAPES[shape]
    lg = logits.double() if logits is not None else hs @ router.double().t()
    ids = torch.topk(lg, s["k"], dim=1).indices
    top = torch.gather(torch.softmax(lg, 1), 1, ids)
    w = top / top.sum(1, keepdim=True)
    out = torch.zeros_like(hs)
    for e in range(s["ne"]):
        t, r = torch.nonzero(ids == e, as_tuple=True)
        if t.numel() == 0:
            continue
        x = hs[t]
        g = _mul(x, _matrix(gu, s["f"], s["d"], seed, 10, layer, e), math_)
        u = _mul(x, _matrix(gu, s["f"], s["d"], seed, 11, layer, e), math_)
        h = torch.nn.functional.silu(g) * u
        out[t] += w[t, r].unsqueeze(1) * _mul(h, _matrix(dn, s["d"], s["f"], seed, 12, layer, e), math_)
    return out, ids, w


def _rope(x, pos, hd, theta):
    """x [n, heads * hd] rotated by pos, the frequency and the angle in 32 bits as the path defines them."""
    i = torch.arange(hd // 2, device=x.device, dtype=torch.float32)
    freq = 1.0 / torch.pow(torch.tensor(theta, device=x.device), 2.0 * i / hd)
    ang = (pos.float().unsqueeze(1) * freq).double()
    c, s = torch.cos(ang).unsqueeze(1), torch.sin(ang).unsqueeze(1)
    v = x.double().view(x.shape[0], -1, hd // 2, 2)
    return torch.stack([v[..., 0] * c - v[..., 1] * s, v[..., 0] * s + v[..., 1] * c], -1).view(x.shape[0], -1, hd)


def _exact_attn(q, k, v, heads, pos_q, theta, window=0):
    """q [n, ..] at positions pos_q over k, v [m, ..] at positions 0 .. m - 1."""
    nh, nkv, hd = HEADS[heads]
    kp = torch.arange(k.shape[0], device=k.device)
    qr, kr, vv = _rope(q, pos_q, hd, theta), _rope(k, kp, hd, theta), v.double().view(v.shape[0], nkv, hd)
    seen = kp.unsqueeze(0) <= pos_q.unsqueeze(1)
    if window:
        seen &= kp.unsqueeze(0) > pos_q.unsqueeze(1) - window
    out = []
    for h in range(nh):
        sc = (qr[:, h] @ kr[:, h * nkv // nh].t()) / math.sqrt(hd)
        out.append(torch.softmax(sc.masked_fill(~seen, -math.inf), 1) @ vv[:, h * nkv // nh])
    return torch.stack(out, 1).reshape(q.shape[0], -1)


def _exact_model(case, seed):
    c, s = MODELS[case["preset"]], SHAPES[case["preset"]]
    nh, nkv, hd = HEADS[c["heads"]]
    d, m = s["d"], c["math"]
    toks = torch.from_numpy(_prompt(case, seed).astype(np.int64)).to(_dev())
    n, T = toks.shape
    pos = torch.arange(T, device=_dev())
    x = _matrix(c["head"], c["vocab"], d, seed, 91, 0)[toks.reshape(-1)]

    def norm(v, i):
        return v / torch.sqrt((v * v).mean(1, keepdim=True) + 1e-5) * _norm_weight(d, seed, i).double()

    for l in range(c["layers"]):
        h = norm(x, l)
        q, k, v = (_mul(h, _matrix(c["proj"], rows, d, seed, 20 + j, l, 0, 0), m)
                   for j, rows in enumerate((nh * hd, nkv * hd, nkv * hd)))
        ctx = torch.cat([_exact_attn(*(t[i * T:(i + 1) * T] for t in (q, k, v)), c["heads"], pos, c["theta"])
                         for i in range(n)])
        x = x + _mul(ctx, _matrix(c["proj"], d, nh * hd, seed, 23, l, 0, 0), m)
        h = norm(x, c["layers"] + l)
        router = torch.from_numpy(_router(case["preset"], seed, False, l)).to(_dev())
        x = x + _exact_moe(case["preset"], c["gu"], c["dn"], m, h, router, None, seed, l)[0]
    x = norm(x, 2 * c["layers"]).view(n, T, d)[:, case["prompt"] - 1:].transpose(0, 1).reshape(-1, d)
    return _mul(x, _matrix(c["head"], c["vocab"], d, seed, 90, 0), m).view(case["steps"] + 1, n, c["vocab"])


def exact(case, seed):
    kind = case["kind"]
    if kind == "moe":
        out, ids, w = _exact_moe(case["shape"], case["gu"], case["dn"], case["math"], _tokens_in(case, seed).double(),
                                 torch.from_numpy(_router(case["shape"], seed, case["skew"])).to(_dev()),
                                 _logits_in(case, seed), seed)
        return dict(out=out, ids=ids, weights=w)
    if kind == "proj":
        return [_mul(_normal((case["tokens"], cols), seed, 30 + j, l).double(), _matrix(qt, rows, cols, seed, 20 + j, l, 0, 0),
                     case["math"])
                for l in range(case["layers"]) for j, (qt, rows, cols) in enumerate(_proj_shapes(case))]
    if kind == "attn_prefill":
        pos = torch.arange(case["tokens"], device=_dev())
        return [_exact_attn(q, k, v, case["heads"], pos, 10000.0)
                for q, k, v in _attn_inputs(case["heads"], case["layers"], case["tokens"], seed, 70)]
    if kind == "attn_decode":
        nkv, hd, win = *HEADS[case["heads"]][1:], case["window"]
        pos, got = torch.tensor([win], device=_dev()), []
        for l, (q, k, v) in enumerate(_attn_inputs(case["heads"], case["layers"], case["seqs"], seed, 70)):
            past = _normal((case["seqs"], win, 2 * nkv * hd), seed, 71, l)
            got.append(torch.cat([_exact_attn(q[i:i + 1], torch.cat([past[i, :, :nkv * hd], k[i:i + 1]]),
                                              torch.cat([past[i, :, nkv * hd:], v[i:i + 1]]), case["heads"], pos, 10000.0, win)
                                  for i in range(case["seqs"])]))
        return got
    return _exact_model(case, seed)
