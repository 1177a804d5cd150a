"""GPU parity of the paths that long prefill chains, small steps of Q8_0 /
Q4_0 models and the backend's single operations take, against the CPU oracle
(models) and a float64 product (operations)."""
import ctypes

import numpy as np
import pytest

import pyoracle as P
from xwfes_amd import ftx
from test_gpu_batch import LOGIT_TOL, random_tree, rel_err_rows, run_batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,heads,kvh,M,npast,tree", [
    (128, 8, 1, 65, 63, False), (128, 8, 2, 129, 0, True), (128, 8, 2, 256, 129, False),
    (64, 16, 2, 255, 5, True), (64, 8, 4, 256, 64, False)])
def test_attention_of_more_than_512_query_rows(gctx, orc, hd, heads, kvh, M, npast, tree):
    """Steps with more than 512 query rows per kv head: several 128-row
    groups, the last ones partly filled, whose last nodes end inside, at and
    past a 64-slot chunk; from an empty context and over one."""
    d = heads * hd
    cfg = P.model_cfg(1, d, heads, kvh, hd, 512, 300, rope_theta=500000.0)
    dts = dict(tok_embd=P.Q8_0, output=P.Q8_0, q=P.Q8_0, k=P.Q8_0, v=P.Q8_0, o=P.Q8_0,
               gate=P.Q8_0, up=P.Q8_0, down=P.Q4_K)
    model = P.make_model(orc, cfg, dts, seed=hd + M)
    rng = np.random.default_rng(M + npast)
    par = random_tree(rng, M, 40, 4) if tree else None
    toks = rng.integers(0, 300, M).tolist()
    (got, want, kv, kvo), = run_batch(gctx, orc, model, [(toks, par, npast, npast + M + 2)], 256)
    assert rel_err_rows(got, want) < LOGIT_TOL
    for a, b in zip(kv, kvo):
        np.testing.assert_allclose(a.astype(np.float32), b.astype(np.float32), rtol=3e-3, atol=3e-3)


def attention_model(orc, hd, heads, kvh, seed, q_std=None, k_std=None):
    """One layer of Q8_0 weights; q_std / k_std: the spread of the q / k
    weights in place of the builder's."""
    d = heads * hd
    cfg = P.model_cfg(1, d, heads, kvh, hd, 512, 300, rope_theta=500000.0)
    dts = dict(tok_embd=P.Q8_0, output=P.Q8_0, q=P.Q8_0, k=P.Q8_0, v=P.Q8_0, o=P.Q8_0,
               gate=P.Q8_0, up=P.Q8_0, down=P.Q4_K)
    model = P.make_model(orc, cfg, dts, seed=seed)
    rng = np.random.default_rng(seed)
    for role, rows, std in (("q", heads * hd, q_std), ("k", kvh * hd, k_std)):
        if std:
            w = (rng.standard_normal((rows, d)) * std).astype(np.float32)
            model["blk.0.%s" % role]["raw"][:] = orc.quantize(w, P.Q8_0).ravel()
    return model


@pytest.mark.parametrize("hd,heads,kvh,M,npast", [(128, 8, 2, 129, 70), (64, 16, 4, 200, 0)])
def test_attention_of_queries_beyond_the_fp16_range(gctx, orc, hd, heads, kvh, M, npast):
    """Query elements of some 1e5 (above fp16's largest value) against keys
    that bring the scores back to ordinary size."""
    model = attention_model(orc, hd, heads, kvh, hd + M, q_std=5000.0, k_std=1e-5)
    toks = np.random.default_rng(M).integers(0, 300, M).tolist()
    (got, want, _, _), = run_batch(gctx, orc, model, [(toks, None, npast, npast + M)], 256)
    assert rel_err_rows(got, want) < LOGIT_TOL


@pytest.mark.parametrize("hd,heads,kvh,M,npast", [(128, 8, 2, 129, 70), (64, 16, 4, 200, 0)])
def test_attention_of_huge_scores(gctx, orc, hd, heads, kvh, M, npast):
    """Scores of some 1e10, whose fp32 neighbours are 1024 apart: one key takes
    all, and no exponent may leave its range.  Rows of a head whose two best
    keys lie within 1e-4 of each other (the fp16 rounding of a key) may take
    either: 7e-4 of them (density of the gap at 0 of some hundred normal
    scores, 7 of their size), 1e-2 of the rows of 8 or 16 heads."""
    model = attention_model(orc, hd, heads, kvh, hd + M, q_std=1.5e6, k_std=10.0)
    toks = np.random.default_rng(M).integers(0, 300, M).tolist()
    (got, want, _, _), = run_batch(gctx, orc, model, [(toks, None, npast, npast + M)], 256)
    assert np.isfinite(want).all() and np.isfinite(got).all()
    err = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    assert (err > LOGIT_TOL).mean() < 0.03


def test_attention_past_a_masked_chunk(gctx, orc):
    """A draft of two roots: the second chain's first 64-slot chunk is all
    masked, and what it sees in the next may score far below 2^-128 of one."""
    model = attention_model(orc, 128, 8, 2, 91, q_std=0.5, k_std=0.5)
    par = [i - 1 for i in range(200)]
    par[100] = -1
    toks = np.random.default_rng(92).integers(0, 300, 200).tolist()
    (got, want, _, _), = run_batch(gctx, orc, model, [(toks, par, 0, 202)], 256)
    assert np.isfinite(want).all() and np.isfinite(got).all()
    err = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    assert np.median(err) < LOGIT_TOL


def test_attention_of_a_long_chain_beside_a_short_one(gctx, orc):
    """Sequences of more than 512 and of at most 16 query rows per kv head in
    one step, in turn: no attention launch takes both."""
    model = attention_model(orc, 128, 16, 2, 77)
    rng = np.random.default_rng(78)
    seqs = [(rng.integers(0, 300, M).tolist(), None, npast, npast + M + 7)
            for M, npast in ((3, 50), (70, 20), (1, 90), (80, 0), (9, 33))]
    for (got, want, kv, kvo) in run_batch(gctx, orc, model, seqs, 256):
        assert rel_err_rows(got, want) < LOGIT_TOL
        for a, b in zip(kv, kvo):
            np.testing.assert_allclose(a.astype(np.float32), b.astype(np.float32), rtol=3e-3, atol=3e-3)


@pytest.mark.parametrize("hd,M,cap,npast", [(64, 65, 66000, 300), (128, 66, 131300, 2000)])
def test_many_rows_over_a_large_cache(gctx, orc, hd, M, cap, npast):
    """More than 512 query rows per kv head over a cache of more than 1024
    attention blocks, whose weights the combine could not hold: the generic
    kernel (steps of fewer rows are refused, test_trace_disarmed_after_failed_launch)."""
    model = attention_model(orc, hd, 8, 1, hd + M)
    toks = np.random.default_rng(M).integers(0, 300, M).tolist()
    (got, want, _, _), = run_batch(gctx, orc, model, [(toks, None, npast, cap)], M)
    assert rel_err_rows(got, want) < LOGIT_TOL


# ---- the backend's single operations ----


def weight(gctx, orc, rng, dt, rows, cols):
    """A quantised weight on the device and its values in float64."""
    raw = orc.quantize((rng.standard_normal((rows, cols)) * 0.02).astype(np.float32), dt)
    values = orc.dequant(raw, dt, cols, rows=rows).reshape(rows, cols)
    return gctx.upload(raw, dt, (cols, rows)), values.astype(np.float64)


def close(got, want, size):
    """|got - want| against `size`, the sum of the products' magnitudes: the
    operands are exact (three bf16 limbs), and sums of blocks in fp32, in chains
    of some 20 additions at most, are off by 20 x 2^-24 of it at worst; 2^-20
    asked for.  A misplaced operand moves a sum by about size / sqrt(terms)."""
    err = np.abs(got - want) / np.maximum(size, 1e-300)
    assert err.max() < 2.0 ** -20, err.max()


@pytest.mark.parametrize("dt", [P.Q4_0, P.Q8_0, P.Q4_K, P.Q6_K])
@pytest.mark.parametrize("M,n_in,blocks", [(1, 1, 1), (3, 33, 2), (16, 257, 3), (17, 31, 5),
                                           (33, 300, 1), (65, 96, 9), (130, 1408, 2),
                                           (1, 1408, 16), (2, 131, 17), (5, 64, 33), (8, 577, 40)])
def test_down_axpy_mfma(gctx, orc, dt, M, n_in, blocks):
    """The column-axpy kernels: the MFMA one at the edges of its token tiles (16,
    32, 64), 32-row slices and 128-column groups, the few-token one (Q8_0,
    Q4_0, up to 8) at those of its 512-column groups, waves' row runs and
    4-row batches; with one split and several; the rows they add to are kept."""
    N = blocks * (256 if dt in (P.Q4_K, P.Q6_K) else 32)
    rng = np.random.default_rng(dt * 1000 + M + n_in)
    t, w = weight(gctx, orc, rng, dt, n_in, N)
    x = rng.standard_normal((M, n_in)).astype(np.float32)
    y0 = (rng.standard_normal((M, N)) * 0.1).astype(np.float32)
    got = gctx.down_axpy(x, t, y0)
    t.free()
    close(got, y0 + x.astype(np.float64) @ w, np.abs(y0) + np.abs(x.astype(np.float64)) @ np.abs(w))


@pytest.mark.parametrize("dt", [P.Q4_0, P.Q8_0, P.Q4_K, P.Q6_K])
def test_down_axpy_special_values(gctx, orc, dt):
    """Infinite, NaN, huge and tiny activations give what a sum of fp32
    products gives; other tokens are untouched by them."""
    rng = np.random.default_rng(5 + dt)
    n_in, N = 70, 512
    t, w = weight(gctx, orc, rng, dt, n_in, N)
    x = rng.standard_normal((6, n_in)).astype(np.float32)
    x[1, 40] = np.inf
    x[2, 3], x[2, 50] = np.inf, -np.inf
    x[3, 69] = np.nan
    x[4] *= np.float32(1e30)
    x[5] *= np.float32(1e-30)
    got = gctx.down_axpy(x, t)
    t.free()
    w32 = w.astype(np.float32)
    with np.errstate(invalid="ignore", over="ignore"):
        want = (x[:, :, None] * w32[None]).astype(np.float64).sum(1)
    keep = [0, 4, 5]
    close(got[keep], want[keep], np.abs(x[keep].astype(np.float64)) @ np.abs(w))
    for m in (1, 2, 3):
        assert np.array_equal(got[m], want[m].astype(np.float32), equal_nan=True)


@pytest.mark.parametrize("dt", [P.Q4_0, P.Q8_0, P.F16, P.F32])
@pytest.mark.parametrize("M,K,N", [(1, 32, 1), (1, 544, 8195), (2, 1056, 37), (3, 512, 300),
                                   (5, 64, 8192), (8, 2080, 66)])
def test_matmul_few_rows(gctx, orc, dt, M, K, N):
    """The few-row kernel: rows of part of a 64-lane stride, whole strides and
    both; one and four output rows per wave, the last wave partly used; every
    activation-row count it is built for and ones between."""
    rng = np.random.default_rng(dt * 100 + M + K + N)
    t, w = weight(gctx, orc, rng, dt, N, K)
    x = rng.standard_normal((M, K)).astype(np.float32)
    got = gctx.matmul(x, t)
    t.free()
    close(got, x.astype(np.float64) @ w.T, np.abs(x.astype(np.float64)) @ np.abs(w).T)


@pytest.mark.parametrize("dt", [P.Q4_0, P.Q8_0, P.Q4_K, P.Q6_K, P.F16, P.F32])
@pytest.mark.parametrize("M,K,N", [(9, 1, 1), (16, 3, 33), (17, 9, 257), (33, 8, 300), (70, 17, 64)])
def test_matmul_many_rows(gctx, orc, dt, M, K, N):
    """More than 8 rows (K in blocks of 32, or of 256 for the K types): the
    edges of 16- and 32-token tiles, 32-row units and 256-element steps, one
    split and several; rows scaled over the fp32 range keep their precision.
    (F32 goes through the few-row kernel in chunks of 8.)"""
    K *= 256 if dt in (P.Q4_K, P.Q6_K) else 32
    rng = np.random.default_rng(dt * 100 + M + K + N)
    t, w = weight(gctx, orc, rng, dt, N, K)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[1] *= np.float32(1e25)
    x[2] *= np.float32(1e-30)
    x[3, K // 2:] *= np.float32(1e-4)
    x[4] = 0
    got = gctx.matmul(x, t)
    t.free()
    assert not got[4].any()
    close(got, x.astype(np.float64) @ w.T, np.abs(x.astype(np.float64)) @ np.abs(w).T)


def outlier(gctx, orc, dt, M, size, down):
    """One activation `size` times the rest of its row, against a weight of zero
    (down: against zeros in every other column): the outputs it adds nothing
    to, held to the magnitudes of the other products alone."""
    rng = np.random.default_rng(dt + M)
    K, N, k0 = 1024, 512, 300
    w = (rng.standard_normal((K, N) if down else (N, K)) * 0.02).astype(np.float32)
    if dt == P.Q4_K:
        w = np.abs(w)  # a minimum of zero, so that zero is one of the block's values
    if down:
        w[k0, ::2] = 0
    else:
        w[:, k0] = 0
    raw = orc.quantize(w, dt)
    v = orc.dequant(raw, dt, w.shape[1], rows=w.shape[0]).reshape(w.shape).astype(np.float64)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[:, k0] = size
    t = gctx.upload(raw, dt, w.shape[::-1])
    got = gctx.down_axpy(x, t) if down else gctx.matmul(x, t)
    t.free()
    v = v if down else v.T
    zero = v[k0] == 0
    assert zero.sum() >= N // 2
    rest = x.astype(np.float64)
    rest[:, k0] = 0
    close(got[:, zero], (rest @ v)[:, zero], (np.abs(rest) @ np.abs(v))[:, zero])


@pytest.mark.parametrize("dt", [P.Q4_0, P.Q8_0, P.Q6_K, P.F16])
@pytest.mark.parametrize("M,size", [(12, 1e8), (40, 1e20)])
def test_matmul_keeps_small_activations_beside_an_outlier(gctx, orc, dt, M, size):
    outlier(gctx, orc, dt, M, size, False)


@pytest.mark.parametrize("down,dt,M", [(False, P.Q4_K, 12), (False, P.Q4_K, 40), (True, P.Q4_K, 4),
                                       (True, P.Q4_K, 40), (True, P.Q4_0, 40), (True, P.Q8_0, 4),
                                       (True, P.Q8_0, 20), (True, P.Q6_K, 20)])
def test_zero_weights_of_a_block_stay_zero(gctx, orc, down, dt, M):
    """Q4_K's zeros are the difference of a scaled integer and a minimum; the
    column-axpy form of every block type."""
    outlier(gctx, orc, dt, M, 1e8, down)


@pytest.mark.parametrize("dt,M", [(P.Q8_0, 4), (P.Q8_0, 12), (P.Q4_0, 12), (P.Q4_K, 12), (P.Q6_K, 12),
                                  (P.F16, 12)])
def test_matmul_special_values(gctx, orc, dt, M):
    """Infinite and NaN activations give what a sum of fp32 products gives,
    and leave the other rows alone."""
    rng = np.random.default_rng(50 + dt)
    K, N = 768, 70
    t, w = weight(gctx, orc, rng, dt, N, K)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[1, 700] = np.inf
    x[2, 3], x[2, 50] = np.inf, -np.inf
    x[3, 69] = np.nan
    got = gctx.matmul(x, t)
    t.free()
    with np.errstate(invalid="ignore"):
        want = (x[:, None, :] * w.astype(np.float32)[None]).astype(np.float64).sum(2)
    keep = [0] + list(range(4, M))
    close(got[keep], want[keep], np.abs(x[keep].astype(np.float64)) @ np.abs(w).T)
    for m in (1, 2, 3):
        assert np.array_equal(got[m], want[m].astype(np.float32), equal_nan=True)


@pytest.mark.parametrize("dt,M,K,IC", [(P.Q4_0, 1, 544, 70), (P.Q8_0, 3, 1024, 4100), (P.F16, 8, 64, 33),
                                       (P.Q4_K, 2, 768, 40), (P.Q6_K, 9, 256, 70), (P.Q4_0, 40, 288, 33)])
def test_expert_chunk_shapes(gctx, orc, dt, M, K, IC):
    """Gate and up rows with SwiGLU through the few-row and the many-row
    kernels, then the column-axpy of the result, added to `out`."""
    rng = np.random.default_rng(dt + M + K + IC)
    (g, wg), (u, wu), (d, wd) = (weight(gctx, orc, rng, dt, IC, K) for _ in range(3))
    x = rng.standard_normal((M, K)).astype(np.float32)
    out = rng.standard_normal((M, K)).astype(np.float32)
    # the rows' device size (Q6_K rows are padded to 16 bytes)
    j = ftx.ExpertJob(x.ctypes.data, 0, g.ptr, u.ptr, d.ptr, dt, 0, M, K, IC, g.nbytes // IC, d.nbytes // IC)
    got = out.copy()
    j.out = got.ctypes.data
    gctx.check(gctx.lib.ftx_expert_chunk(gctx.h, ctypes.byref(j)))
    for t in (g, u, d):
        t.free()
    xg, xu = x.astype(np.float64) @ wg.T, x.astype(np.float64) @ wu.T
    h = xg / (1 + np.exp(-xg)) * xu
    # h itself is a product of two sums: each off by its own size
    ax = np.abs(x.astype(np.float64))
    ah = (ax @ np.abs(wg).T + 1) * (ax @ np.abs(wu).T)
    close(got, out + h @ wd, np.abs(out) + ah @ np.abs(wd))


def test_expert_chunk_in_several_launches(gctx, orc):
    """So many gate / up rows that the tokens go through the GEMM 64 at a time,
    the last launch with fewer."""
    rng = np.random.default_rng(91)
    M, K, IC, dt = 150, 32, 262144, P.Q8_0
    (g, wg), (u, wu), (d, wd) = (weight(gctx, orc, rng, dt, IC, K) for _ in range(3))
    x = rng.standard_normal((M, K)).astype(np.float32)
    got = rng.standard_normal((M, K)).astype(np.float32)
    out = got.astype(np.float64)
    j = ftx.ExpertJob(x.ctypes.data, got.ctypes.data, g.ptr, u.ptr, d.ptr, dt, 0, M, K, IC, g.nbytes // IC,
                      d.nbytes // IC)
    gctx.check(gctx.lib.ftx_expert_chunk(gctx.h, ctypes.byref(j)))
    for t in (g, u, d):
        t.free()
    size = np.abs(out)
    for m in range(M):
        xg, xu = wg @ x[m].astype(np.float64), wu @ x[m].astype(np.float64)
        h = xg / (1 + np.exp(-xg)) * xu
        out[m] += h @ wd
        size[m] += np.abs(h) @ np.abs(wd)
    # 262144 products of a row: the splits' and waves' fp32 chains of some 64
    # additions at most, 64 x 2^-24
    assert (np.abs(got - out) / size).max() < 2.0 ** -18


@pytest.mark.parametrize("dts,d,ff", [("q8_0", 512, 1408), ("q4_0", 256, 544), ("f16", 128, 200),
                                      ("mixed", 384, 512)])
@pytest.mark.parametrize("M", [1, 3, 8])
def test_small_steps_of_stored_types(gctx, orc, dts, d, ff, M):
    """One to eight tokens through models whose projections run on the
    few-row kernel with the RMSNorm in it (one type, and q / k / v of
    different types) and whose ffn_down is Q8_0 / Q4_0 of whole and part
    128-column groups, or F16 on the generic kernel."""
    one = {"q8_0": P.Q8_0, "q4_0": P.Q4_0, "f16": P.F16, "mixed": P.Q8_0}[dts]
    types = dict(tok_embd=P.F32, output=one, q=one, k=one, v=one, o=one, gate=one, up=one, down=one)
    if dts == "mixed":
        types.update(k=P.Q4_0, v=P.F16, o=P.Q4_0)
    cfg = P.model_cfg(2, d, d // 64, max(d // 128, 1), 64, ff, 500, rope_theta=10000.0)
    model = P.make_model(orc, cfg, types, seed=d + M)
    toks = np.random.default_rng(M).integers(0, 500, M).tolist()
    (got, want, kv, kvo), = run_batch(gctx, orc, model, [(toks, None, 21, 40)], 16)
    assert rel_err_rows(got, want) < LOGIT_TOL
    for a, b in zip(kv, kvo):
        np.testing.assert_allclose(a.astype(np.float32), b.astype(np.float32), rtol=3e-3, atol=3e-3)


@pytest.mark.parametrize("q,k,v", [(P.Q4_K, P.Q4_K, P.Q6_K), (P.Q6_K, P.Q8_0, P.Q4_K),
                                   (P.Q4_K, P.Q4_0, P.Q6_K)])
@pytest.mark.parametrize("M", [9, 33, 130])
def test_projections_of_different_types(gctx, orc, q, k, v, M):
    """q / k / v of different types in one projection of more than 8 tokens:
    runs of one type over one operand (two and three launches, their split
    partials side by side), and a Q4_0 between the others, whose operand
    order they do not share; ffn_down Q6_K."""
    dts = dict(tok_embd=P.Q8_0, output=P.Q6_K, q=q, k=k, v=v, o=P.Q6_K, gate=P.Q4_K, up=P.Q4_K,
               down=P.Q6_K)
    cfg = P.model_cfg(2, 1024, 8, 2, 128, 1024, 300, rope_theta=500000.0)
    model = P.make_model(orc, cfg, dts, seed=q + 10 * k + M)
    toks = np.random.default_rng(M + v).integers(0, 300, M).tolist()
    (got, want, _, _), = run_batch(gctx, orc, model, [(toks, None, 30, 30 + M + 3)], 256)
    assert rel_err_rows(got, want) < LOGIT_TOL


@pytest.mark.parametrize("dt", [P.Q8_0, P.Q4_0])
@pytest.mark.parametrize("d,ff,M", [(2048, 520, 1), (2304, 2080, 2), (4096, 2048, 3), (2048, 4128, 8)])
def test_small_steps_over_tiles(gctx, orc, dt, d, ff, M):
    """One to eight tokens of a Q8_0 / Q4_0 model on the re-tiled copies: one
    step per wave, uneven steps and two per wave; a last 16-row tile of 8
    rows (520 gate rows); the head's rows past the last whole tile."""
    dts = dict(tok_embd=P.Q8_0, output=dt, q=dt, k=dt, v=dt, o=dt, gate=dt, up=dt, down=dt)
    cfg = P.model_cfg(1, d, d // 128, max(d // 512, 1) if d != 2304 else 3, 128, ff, 203,
                      rope_theta=500000.0)
    model = P.make_model(orc, cfg, dts, seed=d + ff + M)
    toks = np.random.default_rng(M).integers(0, 203, M).tolist()
    (got, want, kv, kvo), = run_batch(gctx, orc, model, [(toks, None, 50, 70)], 16)
    assert rel_err_rows(got, want) < LOGIT_TOL
    for a, b in zip(kv, kvo):
        np.testing.assert_allclose(a.astype(np.float32), b.astype(np.float32), rtol=3e-3, atol=3e-3)


# ---- scales and activations at the ends of their ranges


def close_or_special(got, want, size):
    """Finite results as close(), the others (infinite, NaN) the same."""
    fin = np.isfinite(want)
    assert np.array_equal(got[~fin], want[~fin].astype(np.float32), equal_nan=True)
    close(got[fin], want[fin], np.broadcast_to(size, want.shape)[fin])


@pytest.mark.parametrize("dt,at", [(P.Q4_0, 0), (P.Q8_0, 0), (P.Q4_K, 0), (P.Q4_K, 2), (P.Q6_K, 208)])
@pytest.mark.parametrize("M", [1, 6, 12])
@pytest.mark.parametrize("down", [False, True])
def test_infinite_and_nan_scales(gctx, orc, dt, at, M, down):
    """A block whose fp16 scale field is infinite or NaN: the products of its
    zero quants are NaN, and so are sums over both signs; the other rows (or
    columns) are untouched.  (Up to 8 rows of the K types' matmul: only the
    rows that hold no such block are looked at.)"""
    rng = np.random.default_rng(7 * dt + at + M)
    K, N = 768, 512
    shape = (K, N) if down else (N, K)
    be, bb = (256, {P.Q4_K: 144, P.Q6_K: 210}[dt]) if dt in (P.Q4_K, P.Q6_K) else (32, {P.Q4_0: 18, P.Q8_0: 34}[dt])
    w32 = (rng.standard_normal(shape) * 0.02).astype(np.float32)
    raw = orc.quantize(w32, dt).reshape(shape[0], shape[1] // be, bb).copy()
    for row, bits in ((5, 0x7C00), (9, 0x7E00)):
        raw[row, 0, at:at + 2] = np.array([bits], np.uint16).view(np.uint8)
    raw = raw.ravel()
    w = orc.dequant(raw, dt, shape[1], rows=shape[0]).reshape(shape)
    x = rng.standard_normal((M, K)).astype(np.float32)
    if down:
        x[:, [5, 9]] = rng.standard_normal((M, 2)) * (rng.random((M, 2)) < 0.8)
    t = gctx.upload(raw, dt, shape[::-1])
    got = gctx.down_axpy(x, t) if down else gctx.matmul(x, t)
    t.free()
    wk = w if down else w.T
    with np.errstate(invalid="ignore"):
        prod = x[:, :, None] * wk[None]
        want, size = prod.astype(np.float64).sum(1), np.abs(prod).astype(np.float64).sum(1)
    if not down and M <= 8 and dt in (P.Q4_K, P.Q6_K):
        assert np.isfinite(got[:, np.isfinite(want[0])]).all()
        return
    close_or_special(got, want, size)


@pytest.mark.parametrize("dt", [P.Q4_0, P.Q8_0])
@pytest.mark.parametrize("M", [1, 4, 20])
def test_down_axpy_large_products(gctx, orc, dt, M):
    """h d beyond the fp32 range where the quant is zero adds nothing."""
    rng = np.random.default_rng(dt + M)
    n_in, N = 40, 512
    w = (rng.standard_normal((n_in, N)) * 500).astype(np.float32)
    w[7, ::2] = 0
    raw = orc.quantize(w, dt)
    v = orc.dequant(raw, dt, N, rows=n_in).reshape(n_in, N)
    x = rng.standard_normal((M, n_in)).astype(np.float32)
    x[0, 7] = 3e38
    t = gctx.upload(raw, dt, (N, n_in))
    got = gctx.down_axpy(x, t)
    t.free()
    with np.errstate(over="ignore"):
        prod = x[:, :, None] * v[None]
        want, size = prod.astype(np.float64).sum(1), np.abs(prod).astype(np.float64).sum(1)
    assert np.isfinite(want[0]).sum() >= N // 2 and np.isinf(want[0]).any()
    close_or_special(got, want, size)


@pytest.mark.parametrize("dt", [P.Q4_0, P.Q8_0, P.Q4_K, P.Q6_K])
@pytest.mark.parametrize("M", [4, 20, 40])
def test_down_axpy_tiny_products(gctx, orc, dt, M):
    """Activations whose products with the weights lie just above the smallest
    normal fp32 number keep their precision."""
    rng = np.random.default_rng(dt + M)
    n_in, N = 200, 512
    t, w = weight(gctx, orc, rng, dt, n_in, N)
    x = (rng.standard_normal((M, n_in)) * 3e-34).astype(np.float32)
    got = gctx.down_axpy(x, t)
    t.free()
    size = np.abs(x.astype(np.float64)) @ np.abs(w)
    # (the sums are kept to 2^-149 at worst)
    assert (np.abs(got - x.astype(np.float64) @ w) < 2.0 ** -20 * size + 2.0 ** -149).all()


@pytest.mark.parametrize("dt,d", [(P.Q8_0, 2048), (P.Q4_0, 2048), (P.Q8_0, 512)])
@pytest.mark.parametrize("M", [1, 5])
def test_small_step_with_an_infinite_head_scale(gctx, orc, dt, d, M):
    """Head rows of one block with an infinite scale: their logits as the
    oracle's (NaN: products of both signs), the others close; over the re-tiled
    copies and over the stored rows."""
    cfg = P.model_cfg(1, d, d // 128, d // 256, 128, 512, 203, rope_theta=10000.0)
    dts = dict(tok_embd=P.Q8_0, output=dt, q=dt, k=dt, v=dt, o=dt, gate=dt, up=dt, down=dt)
    model = P.make_model(orc, cfg, dts, seed=d + M + dt)
    bb = 34 if dt == P.Q8_0 else 18
    rows = model["output"]["raw"].reshape(203, d // 32, bb)
    bad = np.arange(203) % 4 == 1
    rows[bad, 3, :2] = np.array([0x7C00], np.uint16).view(np.uint8)
    toks = np.random.default_rng(M).integers(0, 203, M).tolist()
    (got, want, _, _), = run_batch(gctx, orc, model, [(toks, None, 20, 40)], 8)
    assert np.array_equal(got[:, bad], want[:, bad], equal_nan=True) and np.isnan(want[:, bad]).any()
    assert rel_err_rows(got[:, ~bad], want[:, ~bad]) < LOGIT_TOL


@pytest.mark.parametrize("dt,d", [(P.Q8_0, 2048), (P.Q4_0, 2048), (P.Q8_0, 512), (P.F16, 512)])
def test_small_step_of_a_huge_residual(gctx, orc, dt, d):
    """Rows so large that their squares overflow: the norm's factor is zero and
    every normalised product with it, as in the oracle."""
    cfg = P.model_cfg(1, d, d // 128, d // 256, 128, 512, 203, rope_theta=10000.0)
    dts = dict(tok_embd=P.F32, output=dt, q=dt, k=dt, v=dt, o=dt, gate=dt, up=dt, down=dt)
    model = P.make_model(orc, cfg, dts, seed=d + dt)
    emb = model["tok_embd"]["raw"].view(np.float32)
    emb[:] = np.where(np.random.default_rng(3).random(emb.shape) < 0.5, -3e38, 3e38)
    (got, want, _, _), = run_batch(gctx, orc, model, [([5, 6, 9], None, 0, 16)], 8)
    assert not want.any() and not got.any()


# ---- residual acceptance: its own row statistics


@pytest.mark.parametrize("V", [1, 3, 127, 4095, 4096, 4097, 8194, 20480, 33001])
@pytest.mark.parametrize("off", [0, 4])
def test_residual_statistics_at_chunk_edges(gctx, orc, V, off):
    """Rows that end inside, at and past a 4096-element chunk and a 128-element
    sub-chunk, of any alignment; logits of any size, masked ones (-inf, the
    type's lowest value) among them, a row whose last element is its maximum."""
    rng = np.random.default_rng(V + off)
    M = 6
    rows = (rng.standard_normal((M + 1, V)) * np.array([1, 3, 0.1, 1, 20, 1, 1])[:, None]).astype(np.float32)
    rows[1, V // 3:V // 2] = -np.inf
    rows[3, 2 * V // 3:] = np.finfo(np.float32).min
    rows[2, V - 1] = 9
    rows[4] += 1e4
    q = rng.dirichlet(np.ones(V) * 0.5, size=M).astype(np.float32)
    b, qb = gctx.buffer((M + 1) * V * 4 + 16), gctx.buffer(M * V * 4)
    b.write(rows, off)
    qb.write(q)
    for seed in range(1, 9):
        parents = [-1, -1, 0, 0, 1, 3] if seed % 2 else list(range(-1, M - 1))
        # every other token the target's favourite, the others the draft's
        props = [int(np.argmax(rows[parents[i] + 1] if (i + seed) % 2 else q[i])) for i in range(M)]
        g = gctx.accept(b.ptr + off, b.ptr + off + V * 4, M, V, props, ftx.ACCEPT_RESIDUAL, temp=0.8,
                        rng=seed, parents=parents, q_ptr=qb.ptr)
        o = orc.verify_accept(rows[0], rows[1:], props, P.ACCEPT_RESIDUAL, temp=0.8, seed=seed,
                              parents=parents, q=q)
        assert (g["accepted"], g["bonus"], g["rng"]) == (o["accepted"], o["bonus"], o["rng"]), seed
        # a ratio of sums of V terms in 64 bits, rounded to fp32
        assert abs(g["margin"] - o["margin"]) < 1e-6, seed
    for x in (b, qb):
        x.free()


@pytest.mark.parametrize("d,down,M", [(16384, P.Q8_0, 12), (16640, P.Q8_0, 12), (16640, P.Q6_K, 9), (288, P.Q8_0, 20)])
def test_down_partials_of_wide_and_ragged_rows(gctx, orc, d, down, M):
    """ffn_down on the stored rows of models at both sides of 16384 columns, and
    of rows that are no whole 256: its partials left to the next norm, or added
    at once."""
    dts = dict(tok_embd=P.Q8_0, output=P.Q8_0, q=P.Q8_0, k=P.Q8_0, v=P.Q8_0, o=P.Q8_0, gate=P.Q8_0,
               up=P.Q8_0, down=down)
    cfg = P.model_cfg(2, d, 2, 1, 64, 1024, 60, rope_theta=10000.0)
    model = P.make_model(orc, cfg, dts, seed=d + down)
    toks = np.random.default_rng(M).integers(0, 60, M).tolist()
    (got, want, _, _), = run_batch(gctx, orc, model, [(toks, None, 5, 40)], 32)
    assert rel_err_rows(got, want) < LOGIT_TOL
