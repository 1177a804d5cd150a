"""GPU parity of the paths that long prefill chains, small steps of Q8_0 /
Q4_0 models and the backend's single operations take, against the CPU oracle
(models) and a float64 product (operations)."""
import numpy as np
import pytest

import pyoracle as P
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


# ---- the backend's single operations ----


def weight(gctx, orc, rng, dt, rows, cols):
    """A quantised weight on the device and its values in float64."""
    raw = orc.quantize((rng.standard_normal((rows, cols)) * 0.02).astype(np.float32), dt)
    values = orc.dequant(raw, dt, cols, rows=rows).reshape(rows, cols)
    return gctx.upload(raw, dt, (cols, rows)), values.astype(np.float64)


def close(got, want, terms):
    """Sums of `terms` fp32 products in any order: each rounding is at most
    2^-24 of a partial sum, which random signs keep near the result's size;
    measured 2e-7 of the row's norm, 1e-6 is far from any misplaced operand."""
    err = np.linalg.norm(got - want, axis=1) / np.maximum(np.linalg.norm(want, axis=1), 1e-30)
    assert err.max() < 1e-6, (err.max(), terms)


@pytest.mark.parametrize("dt", [P.Q4_0, P.Q8_0, P.Q4_K, P.Q6_K])
@pytest.mark.parametrize("M,n_in,blocks", [(1, 1, 1), (3, 33, 2), (16, 257, 3), (17, 31, 5),
                                           (33, 300, 1), (65, 96, 9), (130, 1408, 2)])
def test_down_axpy_mfma(gctx, orc, dt, M, n_in, blocks):
    """The column-axpy MFMA kernel at the edges of its token tiles (16, 32, 64),
    32-row slices and 128-column groups, with one split and several; the
    rows it adds to are kept."""
    N = blocks * (256 if dt in (P.Q4_K, P.Q6_K) else 32)
    rng = np.random.default_rng(dt * 1000 + M + n_in)
    t, w = weight(gctx, orc, rng, dt, n_in, N)
    x = rng.standard_normal((M, n_in)).astype(np.float32)
    y0 = (rng.standard_normal((M, N)) * 0.1).astype(np.float32)
    got = gctx.down_axpy(x, t, y0)
    t.free()
    close(got.astype(np.float64), y0 + x.astype(np.float64) @ w, n_in)


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
    for m in (0, 4, 5):
        close(got[m:m + 1].astype(np.float64), want[m:m + 1], n_in)
    for m in (1, 2, 3):
        assert np.array_equal(got[m], want[m].astype(np.float32), equal_nan=True)
