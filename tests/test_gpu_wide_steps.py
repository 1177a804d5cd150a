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
