"""GPU parity of lmx_matvec against the oracle's `dot_row` restatement
(crates/gguf/src/quant.rs:187-271) for every block format the path takes.

Tolerance: max|y - ref| <= 3e-5 * max|ref|: both sum thousands of f32
products, in different orders (the oracle per 32-element sub-block as the
reference does, the GPU per lane then across lanes)."""
import sys

import numpy as np
import pytest

import oracle

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import llmoxide_amd as lmx  # noqa: E402

TYPES = ["q4_k", "q6_k", "q8_0", "f32", "f16", "bf16"]


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def run(name, rows, in_dim, n_tok, seed):
    say(f"matvec {name} rows={rows} in_dim={in_dim} n_tok={n_tok}")
    ty = oracle.QTYPES[name]
    w = oracle.quant_weights(ty, rows, in_dim, seed)
    x = oracle.normal(seed + 50, (n_tok, in_dim))
    ref = oracle.matvec(ty, w, rows, in_dim, x)
    y = lmx.matvec(torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda(), qtype=name, rows=rows,
                   in_dim=in_dim)
    torch.cuda.synchronize()
    got = y.cpu().numpy()
    err = np.abs(got - ref).max()
    assert err <= 3e-5 * np.abs(ref).max(), f"{name}: max err {err} vs max |ref| {np.abs(ref).max()}"


@pytest.mark.parametrize("name", TYPES)
def test_attn_output_shape_decode(name):
    # Qwen3-8B attn_output: 4096 x 4096, one token
    run(name, 4096, 4096, 1, seed=1)


@pytest.mark.parametrize("name", TYPES)
@pytest.mark.parametrize("n_tok", [2, 4, 7])
def test_ragged_rows_and_token_tiles(name, n_tok):
    # rows not a multiple of the 16 a workgroup takes; 7 tokens = two launches
    run(name, 37, 512, n_tok, seed=2 + n_tok)


@pytest.mark.parametrize("name", ["q4_k", "q6_k", "q8_0"])
def test_widest_rows(name):
    run(name, 64, 16384, 1, seed=9)


def test_odd_q6k_block_count_per_row():
    # 3 blocks per row: half the blocks start 2 bytes past a dword boundary
    run("q6_k", 33, 768, 2, seed=10)


@pytest.mark.parametrize("name", ["q4_k", "q6_k", "q8_0"])
@pytest.mark.parametrize("rows,in_dim,n_tok", [(70, 2560, 1), (41, 6400, 1), (41, 12544, 3)])
def test_partial_and_multiple_chunks(name, rows, in_dim, n_tok):
    # Q6_K and Q8_0 rows staged through LDS in 64-unit chunks: 40 units (one
    # partial chunk), 100 units (a full and a partial one) and 196 units
    # (three full chunks and a 4-unit one); odd Q6_K blocks per row put the
    # chunks' windows at every 2-byte offset mod 16.
    run(name, rows, in_dim, n_tok, seed=11 + rows + n_tok)


@pytest.mark.parametrize("name,in_dim", [("f32", 2048), ("f32", 3648), ("f16", 2048), ("f16", 4096), ("f16", 3776),
                                         ("bf16", 2048), ("bf16", 3776)])
@pytest.mark.parametrize("n_tok", [1, 2, 3, 4])
def test_dense_unit_loops(name, in_dim, n_tok):
    # rows of whole 8-unit and 4-unit steps a lane, and of each with single
    # units and a last one that only some lanes have
    run(name, 21, in_dim, n_tok, seed=100 + in_dim + n_tok)


# ---- the matrix-core GEMM (gemm_min_tokens): same bar --
GEMM_TYPES = ["q4_k", "q6_k", "q8_0"]


def run_rows(name, rows, in_dim, n_tok, seed, check_rows):
    """GEMM over the whole matrix, oracle on the listed rows only."""
    say(f"gemm {name} rows={rows} in_dim={in_dim} n_tok={n_tok} checked rows={len(check_rows)}")
    ty = oracle.QTYPES[name]
    w = oracle.quant_weights(ty, rows, in_dim, seed)
    x = oracle.normal(seed + 50, (n_tok, in_dim))
    y = lmx.matvec(torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda(), qtype=name, rows=rows,
                   in_dim=in_dim)
    torch.cuda.synchronize()
    got = y.cpu().numpy()
    rb = oracle.row_bytes(ty, in_dim)
    sub = np.ascontiguousarray(w.reshape(rows, rb)[check_rows])
    ref = oracle.matvec(ty, sub, len(check_rows), in_dim, x)
    err = np.abs(got[:, check_rows] - ref).max()
    assert err <= 3e-5 * np.abs(ref).max(), f"{name}: max err {err} vs max |ref| {np.abs(ref).max()}"
    assert np.all(np.isfinite(got))


@pytest.mark.parametrize("name", GEMM_TYPES)
@pytest.mark.parametrize("n_tok", [16, 64])
def test_gemm_attn_output_shape(name, n_tok):
    # Qwen3-8B attn_output 4096 x 4096 at the GEMM threshold and one token block
    run(name, 4096, 4096, n_tok, seed=20 + n_tok)


@pytest.mark.parametrize("name", GEMM_TYPES)
def test_gemm_prefill_chunk_512(name):
    # the benched shape: a 512-token chunk through attn_output; every token,
    # rows from the first, a middle and the last row block
    rows = list(range(0, 128)) + list(range(2000, 2050)) + list(range(4096 - 130, 4096))
    run_rows(name, 4096, 4096, 512, seed=31, check_rows=rows)


@pytest.mark.parametrize("name,in_dim", [("q4_k", 512), ("q6_k", 768), ("q8_0", 640)])
@pytest.mark.parametrize("rows,n_tok", [(200, 33), (37, 16), (130, 65)])
def test_gemm_ragged_edges(name, in_dim, rows, n_tok):
    # rows and tokens off the tiles; Q6_K with 3 blocks a row puts odd rows 2
    # bytes off a dword; Q8_0 with 20 blocks a row
    run(name, rows, in_dim, n_tok, seed=40 + rows + n_tok)


@pytest.mark.parametrize("in_dim", [128, 384])
def test_gemm_one_and_three_chunks(in_dim):
    # rows of half a 256-weight chunk, and of one and a half
    run("q8_0", 130, in_dim, 70, seed=70 + in_dim)


# (type, rows, in_dim, tokens from which the GEMM runs: gemm_min_tokens)
THRESHOLDS = [("q4_k", 256, 1024, 16), ("q6_k", 7, 2304, 16), ("q6_k", 256, 1024, 9), ("q6_k", 256, 2304, 13), ("q6_k", 40, 4096, 14),
              ("q6_k", 2049, 2304, 9), ("q6_k", 8192, 768, 5), ("q8_0", 7, 1024, 9), ("q8_0", 7, 2304, 16),
              ("q8_0", 256, 1024, 6), ("q8_0", 256, 2304, 8), ("q8_0", 256, 4224, 7), ("q8_0", 2049, 384, 5),
              ("f16", 256, 1024, 9), ("bf16", 256, 1024, 9)]


@pytest.mark.parametrize("name,rows,in_dim,n_min", THRESHOLDS)
def test_matvec_and_gemm_agree_across_the_threshold(name, rows, in_dim, n_min):
    # the last batch that takes the matvec and the first that takes the GEMM
    for n_tok in (n_min - 1, n_min):
        run(name, rows, in_dim, n_tok, seed=60)


@pytest.mark.parametrize("name", GEMM_TYPES)
def test_gemm_x_range(name):
    # x outside f16's comfortable range, per token: large (|x| ~ 1e5, past
    # f16's 65504), tiny (~1e-6, f16 subnormals), and rows whose 128-weight
    # chunks grow or shrink by 11 orders of magnitude along the row (the
    # running per-token scale).  Each token is checked against its own
    # largest |ref|, so tiny tokens need full relative precision.
    rows, in_dim, n_tok = 130, 1024, 64
    say(f"gemm {name} x range rows={rows} in_dim={in_dim} n_tok={n_tok}")
    ty = oracle.QTYPES[name]
    w = oracle.quant_weights(ty, rows, in_dim, 80)
    x = oracle.normal(81, (n_tok, in_dim)).astype(np.float64)
    ramp = np.logspace(-6, 5, in_dim // 128).repeat(128)
    for t in range(n_tok):
        kind = t % 5
        if kind == 1:
            x[t] *= 1e5
        elif kind == 2:
            x[t] *= 1e-6
        elif kind == 3:
            x[t] *= ramp
        elif kind == 4:
            x[t] *= ramp[::-1]
    x = x.astype(np.float32)
    ref = oracle.matvec(ty, w, rows, in_dim, x)
    y = lmx.matvec(torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda(), qtype=name, rows=rows,
                   in_dim=in_dim)
    torch.cuda.synchronize()
    got = y.cpu().numpy()
    assert np.all(np.isfinite(got))
    for t in range(n_tok):
        err = np.abs(got[t] - ref[t]).max()
        scale = np.abs(ref[t]).max()
        assert err <= 3e-5 * scale, f"{name} token {t} (kind {t % 5}): max err {err} vs max |ref| {scale}"


@pytest.mark.parametrize("name,in_dim", [("bf16", 320), ("bf16", 2560), ("f16", 192), ("f16", 1024)])
@pytest.mark.parametrize("rows,n_tok", [(37, 16), (70, 33), (200, 65), (1, 130)])
def test_gemm_dense_edges(name, in_dim, rows, n_tok):
    # dense rows through the GEMM: K ending inside a 256-weight chunk, rows and
    # tokens off the 32- and 64-wide tiles
    run(name, rows, in_dim, n_tok, seed=90 + rows + n_tok)


@pytest.mark.parametrize("name,in_dim", [("q4_k", 768), ("q6_k", 256), ("q6_k", 1280), ("q8_0", 384)])
@pytest.mark.parametrize("rows,n_tok", [(1, 16), (33, 32), (65, 64), (8200, 40), (16500, 17)])
def test_gemm_row_tiles(name, in_dim, rows, n_tok):
    # 32-row tiles beside 32 and 64 tokens, and 64-row ones beside 32 (16500);
    # the last row's bytes end the matrix
    run(name, rows, in_dim, n_tok, seed=120 + rows % 97 + n_tok)


def test_gemm_bf16_weight_range():
    # a chunk of a row is scaled by its own largest weight: rows and chunks of
    # very different sizes, zeros, and a row that falls by 2^-20 along a chunk
    rows, in_dim, n_tok = 40, 512, 20
    rng = np.random.default_rng(7)
    w = rng.standard_normal((rows, in_dim)).astype(np.float32)
    w[1] *= 1e-30
    w[2] *= 1e30
    w[3, 256:] *= 1e-12
    w[4] = 0.0
    w[5] *= np.exp2(-20.0 * np.arange(in_dim) / 256).astype(np.float32)
    bits = (w.view(np.uint32) >> 16).astype(np.uint16)
    w64 = (bits.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    x = oracle.normal(91, (n_tok, in_dim))
    y = lmx.matvec(torch.from_numpy(bits.view(np.uint8).reshape(-1).copy()).cuda(), torch.from_numpy(x).cuda(),
                   qtype="bf16", rows=rows, in_dim=in_dim)
    torch.cuda.synchronize()
    got, ref = y.cpu().numpy().astype(np.float64), x.astype(np.float64) @ w64.T
    for r in range(rows):  # each row against its own scale
        assert np.abs(got[:, r] - ref[:, r]).max() <= 3e-6 * np.abs(ref[:, r]).max(), r


def f64_ref(name, w, rows, in_dim, x):
    """W x in float64 (W as the format's exact values)."""
    W = oracle.dequant(oracle.QTYPES[name], w, rows * in_dim).reshape(rows, in_dim)
    return x.astype(np.float64) @ W.astype(np.float64).T


def gemm(name, w, rows, in_dim, x):
    y = lmx.matvec(torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda(), qtype=name, rows=rows, in_dim=in_dim)
    torch.cuda.synchronize()
    return y.cpu().numpy()


@pytest.mark.parametrize("name", GEMM_TYPES + ["f16", "bf16"])
@pytest.mark.parametrize("n_tok", [21, 49])
def test_gemm_smallest_x(name, n_tok):
    # x whose scale exponent is beyond 100 (below 2^-86), alone, before and
    # after ordinary chunks and zero ones; the x stay normal floats
    rows, in_dim = 70, 1024
    say(f"gemm {name} smallest x n_tok={n_tok}")
    w = oracle.quant_weights(oracle.QTYPES[name], rows, in_dim, 84)
    x = oracle.normal(85, (n_tok, in_dim)).astype(np.float64)
    ends = {0: (1e-30, 1e-30), 1: (1e-27, 1.0), 2: (1.0, 1e-27), 3: (0.0, 1e-30), 4: (1e-30, 0.0),
            5: (1e-35, 1e-20), 6: (1.5 * 2.0 ** -86, 1e4)}
    for t in range(n_tok):
        first, rest = ends[t % 7]
        x[t, :256] *= first
        x[t, 256:] *= rest
    x = x.astype(np.float32)
    got, ref = gemm(name, w, rows, in_dim, x), f64_ref(name, w, rows, in_dim, x)
    for t in range(n_tok):
        err, scale = np.abs(got[t] - ref[t]).max(), np.abs(ref[t]).max()
        assert err <= 3e-5 * scale, f"{name} token {t} (kind {t % 7}): max err {err} vs max |ref| {scale}"


@pytest.mark.parametrize("name", GEMM_TYPES + ["f16", "bf16"])
@pytest.mark.parametrize("n_tok", [20, 70])
def test_gemm_small_x_keeps_its_bits(name, n_tok):
    # the split of x into two f16 parts costs no more at an attention or FFN
    # output's scale than at 1.  Bound: 2^-21 of the result's 2-norm, eight
    # fp32 roundings, for the fp32 sums of 2048 products and 8 to 64 blocks.
    rows, in_dim = 200, 2048
    w = oracle.quant_weights(oracle.QTYPES[name], rows, in_dim, 86)
    x0 = oracle.normal(87, (n_tok, in_dim))
    for rms in (1.0, 0.1, 0.02, 0.006, 3e-5):
        x = x0 * np.float32(rms)
        got, ref = gemm(name, w, rows, in_dim, x), f64_ref(name, w, rows, in_dim, x)
        err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        say(f"gemm {name} n_tok={n_tok} x rms {rms}: {err:.2e}")
        assert err <= 2.0 ** -21, (name, rms, err)


@pytest.mark.parametrize("name", ["f16", "bf16"])
@pytest.mark.parametrize("n_tok", [4, 20, 70])
def test_dense_infinite_and_nan(name, n_tok):
    # products and sums that are infinite or NaN come out as the fp32 matvec
    # (4 tokens) has them, and touch no other token or row
    rows, in_dim = 70, 512
    w = oracle.quant_weights(oracle.QTYPES[name], rows, in_dim, 88).view(np.uint16).reshape(rows, in_dim).copy()
    inf, nan = (0x7C00, 0x7E00) if name == "f16" else (0x7F80, 0x7FC0)
    w[3, 100] = inf
    w[4, 300] = inf | 0x8000
    w[5, [7, 411]] = inf, inf | 0x8000  # inf - inf, where the x agree in sign
    w[6, 90] = nan
    w[8] &= 0x8000                      # 0 times an infinite x
    if name == "bf16":
        w[3, 102:108] = 0x7149          # 1e30 beside the infinite weight
    x = oracle.normal(89, (n_tok, in_dim))
    x[1, 200] = np.inf
    x[2, [30, 31]] = np.inf, -np.inf
    x[3, 511] = np.nan
    if n_tok > 4:
        x[9, 100] = -np.inf             # meets the infinite weight
        x[10, 100] = 0.0                # and 0 does
        x[11] *= np.float32(1e36)       # large beside infinite weights
        x[12, :] = 0.0
        x[12, 5] = np.inf               # before any nonzero x
    w = w.reshape(-1).view(np.uint8)
    got = gemm(name, w, rows, in_dim, x).astype(np.float64)
    W = oracle.dequant(oracle.QTYPES[name], w, rows * in_dim).reshape(rows, in_dim).astype(np.float64)
    with np.errstate(invalid="ignore"):
        ref = np.stack([(W * xt.astype(np.float64)).sum(-1) for xt in x])
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    for t in range(n_tok):
        f = np.isfinite(ref[t])
        if f.any():
            assert np.abs(got[t, f] - ref[t, f]).max() <= 3e-5 * np.abs(ref[t, f]).max(), t


# ---- large grids: 64 tokens x 64 rows, 64 x 128 (the kernel of its own,
# qgemm_big.hip), and dense 32 tokens x 64 rows.  All rows are computed; the
# first, some in the middle and the last are checked.
def some_rows(rows):
    return sorted(set(list(range(140)) + list(range(rows // 2, rows // 2 + 70)) + list(range(rows - 140, rows))))


def run_some(name, rows, in_dim, n_tok, seed, x=None):
    say(f"gemm {name} rows={rows} in_dim={in_dim} n_tok={n_tok}")
    w = oracle.quant_weights(oracle.QTYPES[name], rows, in_dim, seed)
    x = oracle.normal(seed + 50, (n_tok, in_dim)) if x is None else x
    got, pick = gemm(name, w, rows, in_dim, x), some_rows(rows)
    assert np.all(np.isfinite(got))
    sub = np.ascontiguousarray(w.reshape(rows, -1)[pick]).reshape(-1)
    ref = f64_ref(name, sub, len(pick), in_dim, x)
    for t in range(n_tok):
        err, scale = np.abs(got[t, pick] - ref[t]).max(), np.abs(ref[t]).max()
        assert err <= 3e-5 * scale, f"{name} token {t}: max err {err} vs max |ref| {scale}"


@pytest.mark.parametrize("name,in_dim", [("q4_k", 256), ("q4_k", 768), ("q6_k", 256), ("q6_k", 768), ("q8_0", 128),
                                         ("q8_0", 384)])
@pytest.mark.parametrize("rows,n_tok", [
    (16321, 64), (8200, 40), (4100, 190),                # 64 x 64
    (4090, 500), (32641, 33), (32768, 64), (8065, 257),  # 64 x 128, whole and ragged,
    (16400, 40), (3000, 512)])                           # and in grids that leave CUs over
def test_gemm_full_grids(name, in_dim, rows, n_tok):
    run_some(name, rows, in_dim, n_tok, seed=140 + rows % 89 + n_tok)


@pytest.mark.parametrize("name,in_dim", [("f16", 320), ("bf16", 256)])
def test_gemm_dense_full_grid(name, in_dim):
    run_some(name, 16500, in_dim, 17, seed=160)  # 32 tokens x 64 rows


@pytest.mark.parametrize("name", GEMM_TYPES)
@pytest.mark.parametrize("rows,n_tok", [(8200, 40), (32641, 40)])
def test_gemm_full_grids_x_range(name, rows, n_tok):
    # test_gemm_x_range's tokens, and ones below 2^-86, in the tiles of a full grid
    in_dim = 768
    x = oracle.normal(92, (n_tok, in_dim)).astype(np.float64)
    ramp = np.logspace(-6, 5, in_dim // 128).repeat(128)
    kinds = [1.0, 1e5, 1e-6, ramp, ramp[::-1], 1e-30, np.where(np.arange(in_dim) < 256, 1e-27, 1.0),
             np.where(np.arange(in_dim) < 256, 0.0, 1e-30)]
    for t in range(n_tok):
        x[t] *= kinds[t % len(kinds)]
    run_some(name, rows, in_dim, n_tok, seed=170, x=x.astype(np.float32))
