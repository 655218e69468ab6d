"""The split products of several tokens at the edges of their tiles, against
fp64: the direct product (up to 16 tokens, or few rows), the resident and the
tiled one (more tokens, whichever is estimated faster; K in one or several
ranges), and a layer's halves over several sequences, which run on them.

Tolerance: a row is an fp32 sum of exact products in another order than the
reference's, |gpu - fp64| <= 1e-5 sum |w x| (test_gpu_proj.py).  A layer half
that normalises first adds the norm's own rounding, a few 2^-24 of each x:
2e-5; the FFN half chains three products: 8e-5 of the last one's sum."""
import numpy as np
import pytest

import quant_ref as Q
from helpers import device_arrays, log

pytestmark = pytest.mark.gpu

TYPES = [(Q.F32, "f32"), (Q.F16, "f16"), (Q.Q4_0, "q4_0"), (Q.Q8_0, "q8_0"), (Q.Q6_K, "q6_k")]
# direct: one token tile, remainders of rows and waves, groups of four blocks
# that the row does not fill; resident: shares of the tiles, K slices of 4 and
# 8 blocks, two K ranges with an uneven last one; tiled (past 64 tokens): one and
# several K ranges, token and row remainders
SHAPES = [(17, 64, 3), (40, 192, 4), (4112, 1088, 2), (300, 3136, 4), (300, 3136, 5), (9000, 1344, 8),
          (50, 2368, 3), (33, 256, 6), (33, 320, 8), (4112, 256, 16), (9000, 512, 15), (4112, 1024, 17),
          (4200, 2048, 33), (8200, 320, 40), (2064, 4352, 50), (4112, 2560, 193), (8208, 256, 250),
          (6160, 1024, 100), (3000, 4096, 300), (8200, 576, 250), (3000, 64, 200)]


def rows_close(got, raw, x, t, rows, cols, tol, what):
    """got [n][rows] against W . x[i] for every token i."""
    w = Q.dequant(raw, t, rows, cols)
    ref, scale = x.astype(np.float64) @ w.T, np.abs(x).astype(np.float64) @ np.abs(w).T
    err = float(np.max(np.abs(got - ref) / (scale + 1e-30)))
    log(f"    {what}: {err:.2e}")
    assert err <= tol, what


@pytest.mark.parametrize("t,name", TYPES)
@pytest.mark.parametrize("rows,cols,n", SHAPES)
def test_product_edges(W, engines, t, name, rows, cols, n):
    if t == Q.Q6_K and cols % 256:
        pytest.skip("Q6_K rows are whole 256-weight super-blocks")
    eng = engines(1, 64)
    raw = W.make_weights(t, rows, cols, salt=rows + cols)
    x = np.random.default_rng(n + rows).standard_normal((n, cols)).astype(np.float32)
    with device_arrays() as track:
        w, xd = track(eng.array(raw)), track(eng.array(x))
        out = track(eng.array((n + 1, rows)))  # one row more: stays as it was
        guard = np.full((n + 1, rows), 7.25, np.float32)
        out.upload(guard)
        log(f"  product {name} {rows}x{cols}, {n} tokens")
        eng.matmul_batch(out.ptr, w.ptr, xd.ptr, rows, cols, n, t)
        got = out.download()
    assert np.array_equal(got[n], guard[n])
    rows_close(got[:n], raw, x, t, rows, cols, 1e-5, f"{name} {rows}x{cols} x {n}")


@pytest.mark.parametrize("t,name", TYPES)
@pytest.mark.parametrize("n,rows", [(9, 48), (40, 4128)])
def test_product_infinities(W, engines, t, name, n, rows):
    """A token with an infinity, one with the largest float and one with a NaN
    give what fp32 products give (the bf16 pieces of an infinity alone would
    cancel to NaN); the other tokens are untouched by them."""
    infinities(W, engines(1, 64), t, name, n, rows, 256)


# where the tiled product runs: F16 and F32 in one K range, every format but
# Q6_K (which keeps the resident one) in several
@pytest.mark.parametrize("t,name", TYPES)
@pytest.mark.parametrize("n,rows,cols", [(250, 8208, 256), (300, 2064, 4352)])
def test_product_infinities_many_tokens(W, engines, t, name, n, rows, cols):
    infinities(W, engines(1, 64), t, name, n, rows, cols)


# direct: four blocks to an x operand (one subtile by shape) and two (three
# subtiles by shape); resident; tiled in the K ranges of its shape
OPTION_SHAPES = [(2048, 2048, 3), (300, 3136, 4), (11264, 2048, 3), (9000, 1344, 4), (4112, 1024, 33), (2064, 4352, 300),
                 (8208, 256, 250), (11264, 2048, 100)]


@pytest.mark.parametrize("t,name", TYPES)
@pytest.mark.parametrize("rows,cols,n", OPTION_SHAPES)
def test_tiling_options_keep_the_bits(tla, W, engines, t, name, rows, cols, n):
    """Row subtiles and token tiles per workgroup change no bit of a product,
    with K cut as the shape has it; one token tile per workgroup takes more than
    eight workgroups per row group where there are more tiles."""
    if t == Q.Q6_K and cols % 256:
        pytest.skip("Q6_K rows are whole 256-weight super-blocks")
    eng = engines(1, 64)
    raw = W.make_weights(t, rows, cols, salt=rows + cols)
    x = np.random.default_rng(n + rows).standard_normal((n, cols)).astype(np.float32)
    with device_arrays() as track:
        w, xd, out = track(eng.array(raw)), track(eng.array(x)), track(eng.array((n, rows)))

        def product():
            out.upload(np.full((n, rows), np.nan, np.float32))
            eng.matmul_batch(out.ptr, w.ptr, xd.ptr, rows, cols, n, t)
            return out.download()

        base = product()
        for opt, values in ((tla.OPT_SPLIT_ROWS, (1, 2, 4)), (tla.OPT_STREAM_TILES, (1, 3))):
            try:
                for v in values:
                    eng.set_option(opt, v)
                    assert np.array_equal(product().view(np.uint32), base.view(np.uint32)), (opt, v)
            finally:
                eng.set_option(opt, 0)
    rows_close(base, raw, x, t, rows, cols, 1e-5, f"{name} {rows}x{cols} x {n}")


@pytest.mark.parametrize("n,rows,cols", [(12, 2048, 5632), (512, 11264, 2048)])
def test_nan_token_costs_little(W, engines, n, rows, cols):
    """A token with a NaN does not hold up the batch it is in: the product stays
    under three times its time without (1.1 to 1.5 times measured; 10 and 35
    times where a lane walked over the columns for each of the token's sums)."""
    eng = engines(1, 64)
    x = np.random.default_rng(9).standard_normal((n, cols)).astype(np.float32)
    best = []
    with device_arrays() as track:
        w, out, xd = track(eng.array(W.make_weights(Q.Q8_0, rows, cols, salt=3))), track(eng.array((n, rows))), track(eng.array(x))
        for value in (0.5, np.nan):
            x[5, 77] = value
            xd.upload(x)
            times = []
            for _ in range(6):
                eng.event(0)
                for _ in range(5):
                    eng.matmul_batch(out.ptr, w.ptr, xd.ptr, rows, cols, n, Q.Q8_0)
                eng.event(1)
                times.append(eng.elapsed(0, 1))
            best.append(min(times))
    log(f"    {best[0] * 200:.1f} us, with a NaN {best[1] * 200:.1f} us")
    assert best[1] < 3 * best[0]


def infinities(W, eng, t, name, n, rows, cols):
    raw = W.make_weights(t, rows, cols, salt=3)
    x = np.random.default_rng(5).standard_normal((n, cols)).astype(np.float32)
    x[0, 40], x[1, 7], x[2, 200] = np.inf, np.finfo(np.float32).max, np.nan
    with device_arrays() as track:
        w, xd, out = track(eng.array(raw)), track(eng.array(x)), track(eng.array((n, rows)))
        eng.matmul_batch(out.ptr, w.ptr, xd.ptr, rows, cols, n, t)
        got = out.download()
    wf = Q.dequant(raw, t, rows, cols)
    col = wf[:, 40]
    assert np.array_equal(got[0][col > 0], np.full((col > 0).sum(), np.inf, np.float32))
    assert np.array_equal(got[0][col < 0], np.full((col < 0).sum(), -np.inf, np.float32))
    assert np.isnan(got[0][col == 0]).all()
    assert np.isnan(got[2]).all()
    keep = [1] + list(range(3, n))
    rows_close(got[keep], raw, x[keep], t, rows, cols, 1e-5, f"{name} finite tokens")


@pytest.mark.parametrize("t,name", TYPES)
@pytest.mark.parametrize("n", [8, 40])
def test_norm_of_huge_rows(O, W, engines, t, name, n):
    """A finite row whose sum of squares overflows is scaled by zero, as the
    reference's rmsnorm does (the product itself of such a row passes the
    largest float: taken over the unscaled row and multiplied by zero after, it
    would be NaN); a row with an infinity is NaN; the others stay."""
    eng = engines(1, 64, 8, 2)
    embd, kv = 512, 128
    wq, wk, wv = (W.make_weights(t, r, embd, salt=i) for i, r in ((1, embd), (2, kv), (3, kv)))
    x = np.random.default_rng(6).standard_normal((n, embd)).astype(np.float32)
    nw = np.random.default_rng(7).uniform(0.5, 1.5, embd).astype(np.float32)
    x[0] = np.copysign(np.float32(3e38), x[0])
    x[1, 300] = -np.inf
    with np.errstate(all="ignore"):
        xn = np.stack([O.rmsnorm(r, nw, 1e-5) for r in x])
    assert not xn[0].any() and np.isnan(xn[1, 300])
    with device_arrays() as track:
        d = [track(eng.array(a)) for a in (wq, wk, wv, x, nw)]
        q, k, v = (track(eng.array((n, r))) for r in (embd, kv, kv))
        eng.attn_qkv(n, q.ptr, k.ptr, v.ptr, d[3].ptr, d[4].ptr, 1e-5, d[0].ptr, d[1].ptr, d[2].ptr, t)
        for got, raw, rows in ((q.download(), wq, embd), (k.download(), wk, kv), (v.download(), wv, kv)):
            assert not got[0].any()
            assert np.isnan(got[1]).all()
            rows_close(got[2:], raw, xn[2:], t, rows, embd, 2e-5, f"{name} qkv {rows} x {n}")


@pytest.mark.parametrize("t,name", TYPES)
@pytest.mark.parametrize("n", [3, 16, 17, 70, 200])
def test_layer_halves(O, W, engines, t, name, n):
    """tla_attn_qkv (with its rmsnorm), tla_attn_out and tla_ffn_block over n
    sequences: the norm and SwiGLU fused where the shape allows, gate and up
    left in hb as they were before."""
    layer_halves(O, W, engines(1, 64, 8, 2), t, name, n, 768)


# n_ff 2304: W_down in two K ranges from the planes of silu(gate) * up; n_ff 4352,
# F32: gate and up take the tiled product, and a launch of its own writes the planes;
# n_embd 2304: norms of more columns than one pass of a workgroup
@pytest.mark.parametrize("t,name,n,n_head,n_head_kv,n_ff", [
    (Q.Q8_0, "q8_0", 170, 8, 2, 2304), (Q.Q6_K, "q6_k", 170, 8, 2, 2304), (Q.F16, "f16", 170, 16, 4, 4352),
    (Q.F32, "f32", 100, 16, 4, 4352), (Q.Q4_0, "q4_0", 170, 8, 2, 2304), (Q.Q8_0, "q8_0", 40, 36, 12, 768),
    (Q.F16, "f16", 12, 36, 12, 768)])
def test_layer_halves_wide(O, W, engines, t, name, n, n_head, n_head_kv, n_ff):
    layer_halves(O, W, engines(1, 64, n_head, n_head_kv), t, name, n, n_ff)


def layer_halves(O, W, eng, t, name, n, ff):
    embd, kv = eng.cfg.n_embd, 64 * eng.cfg.n_head_kv
    wq, wk, wv = (W.make_weights(t, r, embd, salt=i) for i, r in ((1, embd), (2, kv), (3, kv)))
    wo = W.make_weights(t, embd, embd, salt=4)
    wg, wu = W.make_weights(t, ff, embd, salt=5), W.make_weights(t, ff, embd, salt=6)
    wd = W.make_weights(t, embd, ff, salt=7)
    rg = np.random.default_rng(n)
    x = rg.standard_normal((n, embd)).astype(np.float32)
    nw = rg.uniform(0.5, 1.5, embd).astype(np.float32)
    xn = np.stack([O.rmsnorm(r, nw, 1e-5) for r in x])
    with device_arrays() as track:
        d = {k: track(eng.array(v)) for k, v in
             (("wq", wq), ("wk", wk), ("wv", wv), ("wo", wo), ("wg", wg), ("wu", wu), ("wd", wd), ("x", x), ("nw", nw))}
        q, k, v = (track(eng.array((n, r))) for r in (embd, kv, kv))
        eng.attn_qkv(n, q.ptr, k.ptr, v.ptr, d["x"].ptr, d["nw"].ptr, 1e-5, d["wq"].ptr, d["wk"].ptr, d["wv"].ptr, t)
        for got, raw, rows in ((q, wq, embd), (k, wk, kv), (v, wv, kv)):
            rows_close(got.download(), raw, xn, t, rows, embd, 2e-5, f"{name} qkv {rows} x {n}")
        y = track(eng.array(x))
        eng.attn_out(n, y.ptr, d["wo"].ptr, d["x"].ptr, t)
        rows_close(y.download() - x, wo, x, t, embd, embd, 2e-5, f"{name} out x {n}")
        hb = track(eng.array((n, 2, ff)))
        eng.ffn_block(n, d["x"].ptr, d["nw"].ptr, 1e-5, d["wg"].ptr, d["wu"].ptr, d["wd"].ptr, ff, t, hb.ptr)
        h, got = hb.download(), d["x"].download()
    rows_close(h[:, 0], wg, xn, t, ff, embd, 2e-5, f"{name} gate x {n}")
    rows_close(h[:, 1], wu, xn, t, ff, embd, 2e-5, f"{name} up x {n}")
    g64, u64 = h[:, 0].astype(np.float64), h[:, 1].astype(np.float64)
    act = g64 / (1 + np.exp(-g64)) * u64
    w = Q.dequant(wd, t, embd, ff)
    err = np.abs(got - (x + act @ w.T)) / (np.abs(act) @ np.abs(w).T + np.abs(x))
    log(f"    {name} ffn x {n}: {err.max():.2e}")
    assert err.max() <= 8e-5
