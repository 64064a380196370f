"""attn_prefill_wide_kernel (head_dim 256 and 512) against the oracle at the
edges of its tiles: query counts around the tokens of a workgroup, kv groups
whose packed heads leave a remainder, kv head counts that share XCDs, divide
over them or do neither, key ranges that start and end inside a tile, rings
that wrap inside one, the batch's own rows beside the ring, key splits.

Tolerance: the path's own (tests/helpers.py): P is rounded to f16, everything
else is fp32, whichever way the work is shared out."""
import numpy as np
import pytest

from tests.helpers import AttnCase, assert_close

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import llmoxide_amd as lmx  # noqa: E402


def dev(a, dtype=None):
    t = torch.from_numpy(np.ascontiguousarray(a))
    return (t if dtype is None else t.view(dtype)).cuda()


def check(c, *, base, window=0, bidi=False, scale=None, gate=None):
    print(f"t={c.t} H={c.H} Hkv={c.Hkv} hd={c.hd} base={base} w={window} bidi={bidi} f16={c.q_f16}", flush=True)
    end = base + c.t
    kw = {}
    if window:
        kc, vc = c.ring(window, base)
        kw = dict(k_cur=dev(c.k16[base:end], torch.float16), v_cur=dev(c.v16[base:end], torch.float16))
    else:
        kc, vc = c.k16[:end], c.v16[:end]
    if gate is not None:
        kw["gate"] = dev(gate)
    q = dev(c.q.astype(np.float16)) if c.q_f16 else dev(c.q)
    out = lmx.attention(q, dev(kc, torch.float16), dev(vc, torch.float16), n_heads=c.H, n_kv_heads=c.Hkv,
                        head_dim=c.hd, base_pos=base, window=window, bidi=bidi, scale=scale, **kw)
    torch.cuda.synchronize()
    ref = c.reference(base_pos=base, window=window, bidi=bidi, scale=scale)
    if gate is not None:
        ref = ref / (1.0 + np.exp(-gate.astype(np.float64)))
    assert_close(out.cpu().numpy(), ref)


# (heads, kv heads): 16 and 6 heads packed, one kv head or as many as heads,
# 3 and 5 kv heads (neither dividing the XCDs nor divided by them)
GROUPS = [(16, 1), (6, 3), (4, 4), (5, 5), (8, 2), (16, 8)]


@pytest.mark.parametrize("q_f16", [False, True])
@pytest.mark.parametrize("hd", [256, 512])
@pytest.mark.parametrize("H,Hkv", GROUPS)
def test_head_groups(H, Hkv, hd, q_f16):
    check(AttnCase(H + hd, t=67, H=H, Hkv=Hkv, hd=hd, n_pos=70, q_f16=q_f16), base=3)


@pytest.mark.parametrize("hd", [256, 512])
@pytest.mark.parametrize("t,base", [(9, 0), (9, 118), (63, 1), (64, 0), (65, 63), (129, 64), (130, 700)])
def test_tile_edges(t, base, hd):
    check(AttnCase(t + base, t=t, H=4, Hkv=2, hd=hd, n_pos=base + t), base=base)


@pytest.mark.parametrize("q_f16", [False, True])
@pytest.mark.parametrize("hd", [256, 512])
@pytest.mark.parametrize("window,t,base", [(96, 70, 0), (96, 70, 31), (100, 33, 250), (64, 200, 77), (33, 40, 500)])
def test_rings_with_the_batch_beside(window, t, base, hd, q_f16):
    # rings shorter than a tile, wrapping inside one, and positions of the
    # batch that the ring has not seen
    check(AttnCase(window + t, t=t, H=4, Hkv=2, hd=hd, n_pos=base + t, q_f16=q_f16), base=base, window=window)


@pytest.mark.parametrize("hd", [256, 512])
def test_bidirectional_and_gated(hd):
    c = AttnCase(hd + 1, t=75, H=4, Hkv=2, hd=hd, n_pos=75 + 20)
    gate = np.random.default_rng(5).standard_normal((c.t, c.H * hd)).astype(np.float32)
    check(c, base=20, bidi=True, gate=gate)


@pytest.mark.parametrize("hd", [256, 512])
def test_key_splits(hd):
    # ten tokens over 2100 keys: a workgroup or two, cut into key splits
    check(AttnCase(hd + 2, t=10, H=4, Hkv=1, hd=hd, n_pos=2110), base=2100)


@pytest.mark.parametrize("hd", [256, 512])
def test_scores_that_grow_along_the_keys(hd):
    # every tile raises the running max by far more than the lazy rescale's
    # slack, so each takes the exact path
    c = AttnCase(hd + 3, t=40, H=4, Hkv=2, hd=hd, n_pos=340)
    grow = np.linspace(0.05, 3.0, 340)[:, None]
    c.k16 = (c.kf * grow).astype(np.float16).view(np.uint16)
    c.kf = c.k16.view(np.float16).astype(np.float32)
    check(c, base=300, scale=1.0)


@pytest.mark.parametrize("q_f16", [False, True])
@pytest.mark.parametrize("t,H,Hkv,hd", [
    (15, 4, 2, 256), (16, 4, 2, 256), (17, 4, 2, 256),       # two heads of 16 tokens fill 32 rows; one of 17
    (9, 6, 2, 256), (32, 3, 3, 256), (33, 3, 3, 256), (64, 2, 1, 256), (65, 2, 1, 256),  # and two workgroups of tokens
    (96, 2, 1, 256), (97, 2, 1, 256),
    (9, 4, 1, 512), (16, 2, 1, 512), (17, 2, 1, 512), (32, 3, 3, 512), (33, 3, 3, 512)])
def test_few_rows(t, H, Hkv, hd, q_f16):
    # the form for few rows at its edges, from position 0, inside the second
    # tile and over several
    for base in (0, 50, 333):
        check(AttnCase(t + base + hd, t=t, H=H, Hkv=Hkv, hd=hd, n_pos=base + t, q_f16=q_f16), base=base)


@pytest.mark.parametrize("q_f16", [False, True])
@pytest.mark.parametrize("hd", [256, 512])
def test_few_rows_options(hd, q_f16):
    # a ring with the batch beside it, every query seeing the whole batch, the
    # output gate, and key splits (10 tokens of a head over 3000 keys)
    c = AttnCase(hd + 7, t=20, H=4, Hkv=2, hd=hd, n_pos=220, q_f16=q_f16)
    check(c, base=200, window=90)
    gate = np.random.default_rng(6).standard_normal((c.t, c.H * hd)).astype(np.float32)
    check(c, base=200, bidi=True, gate=gate)
    check(AttnCase(hd + 8, t=10, H=2, Hkv=2, hd=hd, n_pos=3000, q_f16=q_f16), base=2990)
    # scores that grow along the keys: every tile rescales
    c = AttnCase(hd + 9, t=12, H=2, Hkv=2, hd=hd, n_pos=340, q_f16=q_f16)
    c.k16 = (c.kf * np.linspace(0.05, 3.0, 340)[:, None]).astype(np.float16).view(np.uint16)
    c.kf = c.k16.view(np.float16).astype(np.float32)
    check(c, base=328, scale=1.0)
