"""Timed cases of the attention and delta-net hot path: the calls a model's
layers make through llmoxide_amd's entry points, from one decoded token to a
whole prompt.

Each case is a dict of plain values.  Kinds:

* ``attend``   one :func:`llmoxide_amd.attention` call: ``t`` queries at
  positions ``base .. base + t - 1`` over an f16 cache.  ``q16`` queries are f16
  (a caller that converted them), else f32, as the attention prologue leaves
  them.  A windowed chunk keeps positions below ``base`` in a ring of ``window``
  slots and passes its own rows as k_cur / v_cur, as a sliding-window layer
  must.  ``normed`` heads are RMS-normed q and k (Qwen3, Gemma 4), with
  ``scale`` 1.0 where the model uses that.
* ``batched``  one ragged decode step: a query per sequence, each with its own
  cache and length.
* ``delta``    a gated delta-net layer's core: conv front, recurrence (token by
  token below 16 tokens, chunked above), gated norm.
* ``project``  one weight matrix in GGUF block layout times ``t`` tokens.
* ``layer``    a whole attention layer from the hidden states: q, k and v
  projections, prologue (norm, RoPE, KV store), attention, output projection.
"""
import math

import torch

import llmoxide_amd as lmx

DEV = "cuda"

# (n_heads, n_kv_heads, head_dim)
QWEN8B = (32, 8, 128)
SMALL = (16, 8, 128)
GEMMA = (16, 8, 256)
GEMMA4_GLOBAL = (16, 1, 512)

# elements and bytes of a weight block
BLOCKS = {"q4_k": (256, 144), "q6_k": (256, 210), "q8_0": (32, 34), "bf16": (1, 2)}


def _attend(shape, t, base, *, window=0, q16=False, normed=True, scale_one=False, **kw):
    h, hkv, hd = shape
    return dict(kw, kind="attend", t=t, base=base, heads=h, kv_heads=hkv, head_dim=hd, window=window,
                q16=q16, normed=normed, scale=1.0 if scale_one else 1.0 / math.sqrt(hd))


def _batched(n_seq, lens_seed, lo=1024, hi=32768, **kw):
    return dict(kw, kind="batched", n_seq=n_seq, lens_seed=lens_seed, ctx_lo=lo, ctx_hi=hi)


def _project(qtype, rows, in_dim, t, **kw):
    return dict(kw, kind="project", qtype=qtype, rows=rows, in_dim=in_dim, t=t)


def _layer(qtype, t, base, **kw):
    return dict(kw, kind="layer", qtype=qtype, t=t, base=base)


def listed():
    return [
        # the smallest attention call: one token early in a conversation
        _attend(SMALL, 1, 511, name="decode_ctx512"),
        # one token late in a long one, Qwen3-8B's layer
        _attend(QWEN8B, 1, 32767, name="decode_ctx32k"),
        # a serving step over many sequences of mixed lengths
        _batched(32, 3232, name="decode_ragged_b32"),
        # the last few tokens of a prompt cut into chunks, or a short reply to
        # a long conversation
        _attend(QWEN8B, 6, 6144, name="remainder_6_on_6k"),
        # a prompt in one call; q as the prologue leaves it
        _attend(QWEN8B, 2048, 0, name="prefill_2048"),
        # a long document, q already in f16
        _attend(QWEN8B, 8192, 0, q16=True, name="prefill_8192_f16"),
        # a sliding-window layer's chunk in the middle of a prompt, odd sizes
        _attend(GEMMA, 1999, 3001, window=1024, normed=False, name="swa_chunk_1999"),
        # Gemma 4's global layers: 16 heads on one kv head of 512
        _attend(GEMMA4_GLOBAL, 2048, 0, scale_one=True, name="global512_2048"),
        # a delta-net layer over a prompt
        dict(kind="delta", t=4096, name="delta_prefill_4096"),
        # and over one decoded token: three small launches
        dict(kind="delta", t=1, name="delta_decode"),
        # attn_output of a prompt chunk, in the format the reference has a GEMM for
        _project("q6_k", 4096, 4096, 512, name="project_q6k_512"),
        # a whole attention layer over a prompt's later chunk
        _layer("q4_k", 500, 1536, name="layer_chunk_500"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "batched", "remainder", "prefill", "swa", "global512", "delta", "project",
                       "layer"])
    if kind == "decode":
        shape = rng.choice([SMALL, QWEN8B, GEMMA, GEMMA4_GLOBAL])
        window = 1024 if shape == GEMMA and rng.random() < 0.5 else 0
        return _attend(shape, 1, _log(rng, 32, 32768) - 1, window=window, q16=rng.random() < 0.25,
                       scale_one=shape[2] == 512)
    if kind == "batched":
        return _batched(_log(rng, 2, 32), rng.randrange(1 << 20), lo=_log(rng, 64, 1024),
                        hi=_log(rng, 2048, 32768))
    if kind == "remainder":
        return _attend(QWEN8B, rng.randint(2, 15), _log(rng, 128, 16384), q16=rng.random() < 0.25)
    if kind == "prefill":
        t = _log(rng, 16, 6000)
        return _attend(rng.choice([QWEN8B, SMALL]), t, rng.choice([0, _log(rng, 64, 4096)]) if t < 4096 else 0,
                       q16=rng.random() < 0.4)
    if kind == "swa":
        return _attend(GEMMA, _log(rng, 16, 4096), rng.choice([0, _log(rng, 64, 16384)]), window=1024,
                       q16=rng.random() < 0.4, normed=False)
    if kind == "global512":
        return _attend(GEMMA4_GLOBAL, _log(rng, 16, 4096), 0, q16=rng.random() < 0.3, scale_one=True)
    if kind == "delta":
        return dict(kind="delta", t=_log(rng, 1, 4096))
    if kind == "project":
        qtype = rng.choice(sorted(BLOCKS))
        return _project(qtype, _log(rng, 512, 12288), 256 * rng.randint(4, 32), _log(rng, 1, 1024))
    return _layer(rng.choice(["q4_k", "q6_k", "q8_0"]), _log(rng, 1, 1024), _log(rng, 64, 4096))


# ----------------------------------------------------------------- inputs --
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32).to(dtype)


def _normed(x, hd, eps=1e-6):
    h = x.view(x.shape[0], -1, hd)
    return (h * torch.rsqrt((h * h).mean(-1, keepdim=True) + eps)).view(x.shape)


def _lens(case):
    g = torch.Generator()
    g.manual_seed(case["lens_seed"])
    return torch.randint(case["ctx_lo"], case["ctx_hi"] + 1, (case["n_seq"],), generator=g).tolist()


def _weights(g, qtype, rows, in_dim):
    """Random weights of about 0.02 in the GGUF layout."""
    elems, nbytes = BLOCKS[qtype]
    if qtype == "bf16":
        return (0.02 * _randn(g, rows, in_dim)).to(torch.bfloat16).view(torch.uint8).view(-1)
    n = rows * in_dim // elems
    blk = torch.randint(0, 256, (n, nbytes), generator=g, device=DEV, dtype=torch.int32).to(torch.uint8)

    def half(scale):  # a positive f16 per block, within a factor of two of scale
        v = scale * (0.7 + 0.7 * torch.rand((n, 1), generator=g, device=DEV))
        return v.to(torch.float16).view(torch.uint8)

    if qtype == "q4_k":    # d, dmin | 12 scale bytes | 128 quant bytes
        blk[:, 0:2] = half(1e-4)
        blk[:, 2:4] = half(7.5e-4)
    elif qtype == "q6_k":  # 128 ql | 64 qh | 16 scales | d
        blk[:, 208:210] = half(1.5e-5)
    else:                  # d | 32 quants
        blk[:, 0:2] = half(2.7e-4)
    return blk.view(-1)


def _dequant(w, qtype, rows, in_dim):
    """The weights as float64 [rows, in_dim]."""
    if qtype == "bf16":
        return w.view(torch.bfloat16).view(rows, in_dim).double()
    blk = w.view(-1, BLOCKS[qtype][1])

    def half(a):
        return blk[:, a:a + 2].contiguous().view(torch.float16).double()

    if qtype == "q8_0":
        q = blk[:, 2:].contiguous().view(torch.int8).double()
        return (half(0) * q).view(rows, in_dim)
    if qtype == "q4_k":
        b = blk[:, 4:16].int()
        lo, hi = b[:, 0:4], b[:, 4:8]
        sc = torch.cat([lo & 63, (b[:, 8:12] & 15) | ((lo >> 6) << 4)], 1)
        mn = torch.cat([hi & 63, (b[:, 8:12] >> 4) | ((hi >> 6) << 4)], 1)
        qs = blk[:, 16:].int().view(-1, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).view(-1, 8, 32)
        return (half(0).unsqueeze(2) * sc.unsqueeze(2) * q - half(2).unsqueeze(2) * mn.unsqueeze(2)).view(rows, in_dim)
    ql = blk[:, 0:128].int().view(-1, 2, 2, 32)       # half, l / 32, l % 32
    qh = blk[:, 128:192].int().view(-1, 2, 1, 32)
    nib = torch.cat([ql & 15, ql >> 4], 2)            # half, quarter, l
    sh = torch.tensor([0, 2, 4, 6], device=w.device, dtype=torch.int32).view(1, 1, 4, 1)
    q = (nib | (((qh >> sh) & 3) << 4)) - 32
    sc = blk[:, 192:208].contiguous().view(torch.int8).double().view(-1, 16, 1)
    return (half(208).unsqueeze(2) * sc * q.reshape(-1, 16, 16).double()).view(rows, in_dim)


def _prepare_attend(case, seed):
    g = _gen(seed)
    t, base, hd, w = case["t"], case["base"], case["head_dim"], case["window"]
    kv_dim = case["kv_heads"] * hd
    q = _randn(g, t, case["heads"] * hd)
    n = base + t
    k, v = _randn(g, n, kv_dim), _randn(g, n, kv_dim, dtype=torch.float16)
    if case["normed"]:
        q, k = _normed(q, hd), _normed(k, hd)
    k = k.half()
    s = dict(q=q.half() if case["q16"] else q, out=torch.empty((t, case["heads"] * hd), device=DEV),
             ws=lmx.Workspace(), cur={})
    if w:
        # a batch's own rows beside the ring; a single token is stored first
        stored = n if t == 1 else base
        ring = [torch.zeros((w, kv_dim), dtype=torch.float16, device=DEV) for _ in range(2)]
        pos = torch.arange(max(0, stored - w), stored, device=DEV)
        for r, src in zip(ring, (k, v)):
            r[pos % w] = src[pos]
        if t > 1:
            s["cur"] = dict(k_cur=k[base:].contiguous(), v_cur=v[base:].contiguous())
        s["k"], s["v"] = ring
    else:
        s["k"], s["v"] = k, v
    s["args"] = dict(n_heads=case["heads"], n_kv_heads=case["kv_heads"], head_dim=hd, base_pos=base,
                     window=w, scale=case["scale"])
    return s


def _prepare_batched(case, seed):
    g = _gen(seed)
    h, hkv, hd = QWEN8B
    lens = _lens(case)
    ks = [_randn(g, n, hkv * hd, dtype=torch.float16) for n in lens]
    vs = [_randn(g, n, hkv * hd, dtype=torch.float16) for n in lens]
    return dict(q=_randn(g, len(lens), h * hd), caches=lmx.BatchedCaches(ks, vs), ks=ks, vs=vs,
                ctx=torch.tensor(lens, dtype=torch.int32, device=DEV), max_ctx=max(lens),
                out=torch.empty((len(lens), h * hd), device=DEV), ws=lmx.Workspace())


# Qwen3.5's delta-net layer
VH, KH, SD, TAPS = 32, 16, 128, 4
KEY_DIM, D_INNER = KH * SD, VH * SD
CONV_DIM = 2 * KEY_DIM + D_INNER


def _prepare_delta(case, seed):
    g = _gen(seed)
    t = case["t"]
    return dict(t=t, x=_randn(g, t, CONV_DIM), taps=0.5 * _randn(g, CONV_DIM, TAPS),
                window=_randn(g, TAPS - 1, CONV_DIM), alpha=_randn(g, t, VH), beta=_randn(g, t, VH),
                state=0.05 * _randn(g, VH, SD, SD), ssm_a=torch.full((VH,), -1.0, device=DEV),
                dt=torch.zeros(VH, device=DEV), z=_randn(g, t, D_INNER),
                w=1.0 + 0.1 * _randn(g, SD), conv=torch.empty((t, CONV_DIM), device=DEV),
                out=torch.empty((t, D_INNER), device=DEV), ws=lmx.Workspace())


def _prepare_project(case, seed):
    g = _gen(seed)
    return dict(w=_weights(g, case["qtype"], case["rows"], case["in_dim"]), x=_randn(g, case["t"], case["in_dim"]),
                y=torch.empty((case["t"], case["rows"]), device=DEV),
                args=dict(qtype=case["qtype"], rows=case["rows"], in_dim=case["in_dim"]))


HIDDEN = 4096
ROPE_BASE = 1e6


def _layer_mats():
    h, hkv, hd = QWEN8B
    return {"q": (h * hd, HIDDEN), "k": (hkv * hd, HIDDEN), "v": (hkv * hd, HIDDEN), "o": (HIDDEN, h * hd)}


def _prepare_layer(case, seed):
    g = _gen(seed)
    h, hkv, hd = QWEN8B
    t, base, n = case["t"], case["base"], case["base"] + case["t"]
    s = dict(x=_randn(g, t, HIDDEN), ws=lmx.Workspace(), qg=1.0 + 0.1 * _randn(g, hd),
             kg=1.0 + 0.1 * _randn(g, hd), base=base, qtype=case["qtype"],
             kc=torch.zeros((n, hkv * hd), dtype=torch.float16, device=DEV),
             vc=torch.zeros((n, hkv * hd), dtype=torch.float16, device=DEV),
             attn=torch.empty((t, h * hd), device=DEV))
    s["kc"][:base] = _normed(_randn(g, base, hkv * hd), hd).half()
    s["vc"][:base] = _randn(g, base, hkv * hd, dtype=torch.float16)
    for name, (rows, in_dim) in _layer_mats().items():
        s["w" + name] = _weights(g, case["qtype"], rows, in_dim)
        s["y" + name] = torch.empty((t, rows), device=DEV)
    return s


def prepare(case, seed):
    return {"attend": _prepare_attend, "batched": _prepare_batched, "delta": _prepare_delta,
            "project": _prepare_project, "layer": _prepare_layer}[case["kind"]](case, seed) | {"case": case}


# -------------------------------------------------------------------- runs --
def run(state):
    s, kind = state, state["case"]["kind"]
    if kind == "attend":
        return lmx.attention(s["q"], s["k"], s["v"], out=s["out"], workspace=s["ws"], **s["args"], **s["cur"])
    if kind == "batched":
        h, hkv, hd = QWEN8B
        return lmx.attention_decode_batched(s["q"], s["caches"], s["ctx"], max_ctx=s["max_ctx"], n_heads=h,
                                            n_kv_heads=hkv, head_dim=hd, n_slots=s["max_ctx"], out=s["out"],
                                            workspace=s["ws"])
    if kind == "delta":
        conv = lmx.delta_front(s["x"], s["taps"], s["window"], s["conv"], key_dim=KEY_DIM, s_dim=SD)
        if s["t"] < 16:
            lmx.delta_recur(conv, s["alpha"], s["beta"], s["state"], s["ssm_a"], s["dt"], n_vh=VH, n_kh=KH,
                            s_dim=SD, out=s["out"])
        else:
            lmx.delta_chunked(conv, s["alpha"], s["beta"], s["state"], s["ssm_a"], s["dt"], n_vh=VH, n_kh=KH,
                              s_dim=SD, out=s["out"], workspace=s["ws"])
        lmx.delta_back(s["out"], s["z"], s["w"], n_vh=VH, s_dim=SD)
        return s["out"], s["state"], s["window"]
    if kind == "project":
        return lmx.matvec(s["w"], s["x"], y=s["y"], **s["args"])
    h, hkv, hd = QWEN8B
    for name, (rows, in_dim) in _layer_mats().items():
        if name != "o":
            lmx.matvec(s["w" + name], s["x"], qtype=s["qtype"], rows=rows, in_dim=in_dim, y=s["y" + name])
    lmx.attn_prologue(s["yq"], s["yk"], s["yv"], s["kc"], s["vc"], n_heads=h, n_kv_heads=hkv, head_dim=hd,
                      base_pos=s["base"], rope_base=ROPE_BASE, q_gain=s["qg"], k_gain=s["kg"])
    lmx.attention(s["yq"], s["kc"], s["vc"], n_heads=h, n_kv_heads=hkv, head_dim=hd, base_pos=s["base"],
                  out=s["attn"], workspace=s["ws"])
    y = lmx.matvec(s["wo"], s["attn"], qtype=s["qtype"], rows=HIDDEN, in_dim=h * hd, y=s["yo"])
    return y, s["kc"][s["base"]:], s["vc"][s["base"]:]


# ------------------------------------------------------------------- work --
def _pairs(t, base, window):
    if not window:
        return t * base + t * (t + 1) // 2
    return sum(min(base + i + 1, window) for i in range(t))


def _attend_work(t, base, h, hkv, hd, window, q_bytes):
    keys = base + t if not window else min(base + t, t + window - 1)
    return dict(bytes=2 * 2 * keys * hkv * hd + t * h * hd * (q_bytes + 4),
                flops=4 * hd * h * _pairs(t, base, window))


def _project_work(qtype, rows, in_dim, t):
    elems, nbytes = BLOCKS[qtype]
    return dict(bytes=rows * in_dim // elems * nbytes + 4 * t * (rows + in_dim), flops=2 * rows * in_dim * t)


def work(case):
    kind = case["kind"]
    if kind == "attend":
        return _attend_work(case["t"], case["base"], case["heads"], case["kv_heads"], case["head_dim"],
                            case["window"], 2 if case["q16"] else 4)
    if kind == "batched":
        h, hkv, hd = QWEN8B
        lens = _lens(case)
        return dict(bytes=sum(2 * 2 * n * hkv * hd for n in lens) + 8 * len(lens) * h * hd,
                    flops=4 * hd * h * sum(lens))
    if kind == "delta":
        t = case["t"]
        # x, z, alpha, beta in; out; state and window in and out; the
        # recurrence's decay, two matrix-vector products and rank-one update
        return dict(bytes=4 * (t * (CONV_DIM + 2 * D_INNER + 2 * VH) + 2 * VH * SD * SD
                               + (2 * (TAPS - 1) + TAPS) * CONV_DIM),
                    flops=t * (VH * SD * SD * 7 + 2 * TAPS * CONV_DIM))
    if kind == "project":
        return _project_work(case["qtype"], case["rows"], case["in_dim"], case["t"])
    h, hkv, hd = QWEN8B
    t, base = case["t"], case["base"]
    mats = [_project_work(case["qtype"], r, c, t) for r, c in _layer_mats().values()]
    att = _attend_work(t, base, h, hkv, hd, 0, 4)
    # x in, y out, the weights, and the cache rows read and stored
    weights = sum(r * c // BLOCKS[case["qtype"]][0] * BLOCKS[case["qtype"]][1] for r, c in _layer_mats().values())
    return dict(bytes=weights + 8 * t * HIDDEN + 4 * hkv * hd * (base + 2 * t),
                flops=att["flops"] + sum(m["flops"] for m in mats))


# Relative errors a correct implementation may show, about four times what was
# measured against float64: 2e-7 to 3e-7 where products and sums are 32-bit
# (decode, projections, the delta recurrence), 1e-4 to 2.1e-4 where the softmax
# weights or the new cache rows are rounded to f16, 2e-5 to 3e-5 at head_dim
# 512 (scale 1.0: few keys carry the weight), 6.5e-6 for the chunked delta
# rule's split bf16 products.
def tolerance(case):
    kind = case["kind"]
    if kind == "attend":
        if case["t"] > 8:
            return {"rel": 8.5e-4}
        return {"rel": 1.2e-4 if case["head_dim"] == 512 else 1.5e-6}
    if kind in ("batched", "project"):
        return {"rel": 1.5e-6}
    if kind == "delta":
        return {"rel": 2.6e-5 if case["t"] >= 16 else 1e-6}
    return {"rel": 8.5e-4}


# ------------------------------------------------------------------ exact --
def _exact_attention(q, k, v, *, base, heads, kv_heads, hd, window, scale):
    """q [t, H*hd], k and v [base + t, Hkv*hd], float64."""
    t, n = q.shape[0], k.shape[0]
    out = torch.empty_like(q)
    rows = max(1, min(t, (1 << 26) // n))
    for h in range(heads):
        c = (h // (heads // kv_heads)) * hd
        kh, vh = k[:, c:c + hd].contiguous(), v[:, c:c + hd].contiguous()
        for i in range(0, t, rows):
            j = min(t, i + rows)
            lo = max(0, base + i + 1 - window) if window else 0
            s = scale * (q[i:j, h * hd:(h + 1) * hd] @ kh[lo:base + j].t())
            pos = torch.arange(base + i, base + j, device=q.device).view(-1, 1)
            key = torch.arange(lo, base + j, device=q.device).view(1, -1)
            hide = key > pos
            if window:
                hide |= key <= pos - window
            out[i:j, h * hd:(h + 1) * hd] = torch.softmax(s.masked_fill_(hide, -math.inf), -1) @ vh[lo:base + j]
    return out


def _exact_attend(case, seed):
    s = _prepare_attend(case, seed)
    t, base, w = case["t"], case["base"], case["window"]
    if w:
        n = base + t
        pos = torch.arange(n, device=DEV)
        k, v = s["k"][pos % w].double(), s["v"][pos % w].double()
        if t > 1:
            k[base:], v[base:] = s["cur"]["k_cur"].double(), s["cur"]["v_cur"].double()
    else:
        k, v = s["k"].double(), s["v"].double()
    return _exact_attention(s["q"].double(), k, v, base=base, heads=case["heads"], kv_heads=case["kv_heads"],
                            hd=case["head_dim"], window=w, scale=case["scale"])


def _exact_batched(case, seed):
    s = _prepare_batched(case, seed)
    h, hkv, hd = QWEN8B
    return torch.cat([_exact_attention(s["q"][i:i + 1].double(), k.double(), v.double(), base=k.shape[0] - 1, heads=h,
                                       kv_heads=hkv, hd=hd, window=0, scale=1.0 / math.sqrt(hd))
                      for i, (k, v) in enumerate(zip(s["ks"], s["vs"]))])


def _exact_delta(case, seed):
    s = _prepare_delta(case, seed)
    t = case["t"]
    full = torch.cat([s["window"], s["x"]]).double()
    taps = s["taps"].double()
    c = sum(full[j:j + t] * taps[:, j] for j in range(TAPS))
    c = c * torch.sigmoid(c)
    qk = c[:, :2 * KEY_DIM].view(t, 2 * KH, SD)
    qk = qk / qk.norm(dim=-1, keepdim=True).clamp_min(1e-6)
    rep = torch.arange(VH, device=DEV) % KH
    q, k = qk[:, :KH][:, rep], qk[:, KH:][:, rep]
    v = c[:, 2 * KEY_DIM:].view(t, VH, SD)
    g = torch.exp(s["ssm_a"].double() * torch.nn.functional.softplus(s["alpha"].double() + s["dt"].double()))
    b = torch.sigmoid(s["beta"].double())
    S = s["state"].double()
    o = torch.empty((t, VH, SD), dtype=torch.float64, device=DEV)
    for i in range(t):
        S = S * g[i].view(VH, 1, 1)
        d = b[i].view(VH, 1) * (v[i] - (S * k[i].unsqueeze(1)).sum(-1))
        S = S + d.unsqueeze(2) * k[i].unsqueeze(1)
        o[i] = (S * q[i].unsqueeze(1)).sum(-1) / math.sqrt(SD)
    z = s["z"].double().view(t, VH, SD)
    o = o * torch.rsqrt((o * o).mean(-1, keepdim=True) + 1e-6) * s["w"].double() * z * torch.sigmoid(z)
    return o.view(t, D_INNER), S, full[-(TAPS - 1):].clone()


def _exact_layer(case, seed):
    s = _prepare_layer(case, seed)
    h, hkv, hd = QWEN8B
    t, base = case["t"], case["base"]
    mats = {n: _dequant(s["w" + n], case["qtype"], r, c) for n, (r, c) in _layer_mats().items()}
    x = s["x"].double()
    ang = torch.arange(base, base + t, device=DEV, dtype=torch.float64).view(-1, 1) * \
        ROPE_BASE ** (-torch.arange(0, hd, 2, device=DEV, dtype=torch.float64) / hd)
    cos, sin = ang.cos().unsqueeze(1), ang.sin().unsqueeze(1)

    def rope_norm(y, gain):
        y = y.view(t, -1, hd)
        y = y * torch.rsqrt((y * y).mean(-1, keepdim=True) + 1e-6) * gain.double()
        a, b = y[..., :hd // 2], y[..., hd // 2:]
        return torch.cat([a * cos - b * sin, a * sin + b * cos], -1).reshape(t, -1)

    q = rope_norm(x @ mats["q"].t(), s["qg"])
    k = rope_norm(x @ mats["k"].t(), s["kg"])
    v = x @ mats["v"].t()
    # the cache holds f16
    kc = torch.cat([s["kc"][:base].double(), k.half().double()])
    vc = torch.cat([s["vc"][:base].double(), v.half().double()])
    a = _exact_attention(q, kc, vc, base=base, heads=h, kv_heads=hkv, hd=hd, window=0, scale=1.0 / math.sqrt(hd))
    return a @ mats["o"].t(), k, v


def exact(case, seed):
    kind = case["kind"]
    if kind == "project":
        s = _prepare_project(case, seed)
        return s["x"].double() @ _dequant(s["w"], case["qtype"], case["rows"], case["in_dim"]).t()
    return {"attend": _exact_attend, "batched": _exact_batched, "delta": _exact_delta,
            "layer": _exact_layer}[kind](case, seed)
