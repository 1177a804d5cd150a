"""The work that a user of this library has it do, as cases to time and compare.

Two kinds of user program stand behind them.  A speculative-decoding engine
keeps the whole model resident and calls the verify step (one token, an
8-token draft, a draft tree, several sequences at once), the prefill of a
prompt and the acceptance of a draft.  An engine that keeps its own graph
calls the backend's single operations (matmul, down_axpy, expert_chunk) with
its own activations.  Sizes are those of bench.py's workloads (the tiny
reference model, Llama-3-8B / 3.2-1B / 3-70B and Mixtral-8x7B shapes); the
deep models run a few of their layers, except one whole 32-layer step.

listed() / draw(rng): the cases; prepare(case, seed): a program's state;
run(state): one pass; exact(case, seed): the same outputs from 64-bit torch.

Weights are synthetic GGUF blocks made here (quantised values of a normal
distribution, block scales that vary by 20 %), so that exact() needs nothing
of the library.
"""
import math

import numpy as np
import torch

from xwfes_amd import ftx

DEV = "cuda"
Q4_0, Q8_0, Q4_K, Q6_K, F16, F32 = ftx.Q4_0, ftx.Q8_0, ftx.Q4_K, ftx.Q6_K, ftx.F16, ftx.F32
TYPES = {"q4_0": Q4_0, "q8_0": Q8_0, "q4_k": Q4_K, "q6_k": Q6_K, "f16": F16, "f32": F32}
STD = 0.02  # of the weights

TINY = dict(layers=4, d=512, heads=8, kv_heads=8, hd=64, ff=1408, vocab=32000, theta=1e4)
LLAMA_1B = dict(layers=4, d=2048, heads=32, kv_heads=8, hd=64, ff=8192, vocab=32000, theta=5e5)
LLAMA_8B = dict(layers=4, d=4096, heads=32, kv_heads=8, hd=128, ff=14336, vocab=32000, theta=5e5)
LLAMA_70B = dict(layers=2, d=8192, heads=64, kv_heads=8, hd=128, ff=28672, vocab=32000, theta=5e5)
MIXTRAL = dict(layers=2, d=4096, heads=32, kv_heads=8, hd=128, ff=14336, vocab=32000, theta=1e6,
               experts=8, used=2)


def listed():
    return [
        # the smallest call: one decode step of the reference's own 4-layer
        # Q4_0 model after its 128-token prompt
        dict(name="step-tiny-q4_0", kind="verify", mix="q4_0", M=1, ctx=129, seqs=1, tree=0, **TINY),
        # the engine's other per-round call: an 8-token draft's acceptance by
        # the ratio test over a 128k vocabulary, with the sampled bonus token
        dict(name="accept-ratio-8", kind="accept", M=8, V=128256, tree=0, temp=0.8),
        # acceptance of a 52-node draft tree by residual resampling
        dict(name="accept-tree-52", kind="accept", M=52, V=128256, tree=4, temp=0.8),
        # one projection of a decode step for an engine that keeps its own
        # graph: host activations in, host activations out
        dict(name="matmul-host-1-q8_0", kind="matmul", dt="q8_0", M=1, K=4096, N=4096, host=1),
        # the same engine with device activations: a draft tree's (or a short
        # prompt's) gate projection
        dict(name="matmul-48-q4_k", kind="matmul", dt="q4_k", M=48, K=4096, N=14336, host=0),
        # one expert over the tokens routed to it
        dict(name="expert-24-q4_0", kind="expert", dt="q4_0", M=24, K=4096, IC=14336, host=0),
        # a decode step of a Q8_0 model (a common file type) at context 2048
        dict(name="step-8b-q8_0", kind="verify", mix="q8_0", M=1, ctx=2048, seqs=1, tree=0,
             **LLAMA_8B),
        # the flagship: an 8-token draft against a whole 32-layer Q4_K_M model
        dict(name="verify8-8b-q4_k_m", kind="verify", mix="q4_k_m", M=8, ctx=2048, seqs=1, tree=0,
             **dict(LLAMA_8B, layers=32, vocab=128256)),
        # a 32-node draft tree at context 4096, Q8_0 attention, Q4_K FFN
        dict(name="tree32-8b-q8attn", kind="verify", mix="q8attn", M=32, ctx=4096, seqs=1, tree=4,
             **LLAMA_8B),
        # four sequences of 8-token drafts through a mixture of experts
        dict(name="batch4x8-mixtral-q4_0", kind="verify", mix="q4_0", M=8, ctx=1024, seqs=4, tree=0,
             **MIXTRAL),
        # a 700-token prompt in chains of 256
        dict(name="prefill-700-8b-q4_k_m", kind="prefill", mix="q4_k_m", M=700, chunk=256,
             **LLAMA_8B),
        # the widest step: four 64-node trees at context 8192 on 70B layers
        dict(name="tree4x64-70b-q4_k", kind="verify", mix="q4_k", M=64, ctx=8192, seqs=4, tree=4,
             **LLAMA_70B),
    ]


def _log_int(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.choice(["verify", "verify", "verify", "matmul", "matmul", "down", "expert",
                       "prefill", "accept"])
    if kind == "accept":
        tree = rng.choice([0, 4])
        return dict(kind=kind, M=_log_int(rng, 1, 16) if not tree else rng.randint(4, 64),
                    V=rng.randint(30000, 160000), tree=tree, temp=rng.choice([0.6, 0.8, 1.0]))
    if kind in ("matmul", "down", "expert"):
        dt = rng.choice(["q4_0", "q8_0", "q4_k", "q6_k", "f16"])
        # whole blocks along a row: 32 elements, 256 for the K types
        step = 256 if dt in ("q4_k", "q6_k") else 32
        cols = step * max(1, _log_int(rng, 512, 8192) // step)
        rows = _log_int(rng, 256, 14336)
        M = _log_int(rng, 1, 256)
        c = dict(kind=kind, dt=dt, M=M, host=int(rng.random() < 0.25))
        if kind == "matmul":
            c.update(K=cols, N=rows)
        elif kind == "down":
            c.update(n_in=rows, N=cols)
        else:
            c.update(K=cols, IC=rows, M=_log_int(rng, 1, 64))
        return c
    shape = dict(rng.choice([TINY, LLAMA_1B, LLAMA_8B, LLAMA_8B]))
    mixes = ["q4_0", "q8_0", "f16"] if shape["d"] == 512 else ["q4_0", "q8_0", "q4_k", "q4_k_m",
                                                               "q8attn"]
    mix = rng.choice(mixes)
    shape["layers"] = rng.randint(1, 4)
    if kind == "prefill":
        return dict(kind=kind, mix=mix, M=_log_int(rng, 9, 700), chunk=rng.choice([64, 128, 256]),
                    **shape)
    seqs = rng.choice([1, 1, 1, 2, 4])
    tree = rng.choice([0, 0, 4])
    M = _log_int(rng, 1, 16) if not tree else rng.randint(4, 64)
    return dict(kind="verify", mix=mix, M=M, ctx=_log_int(rng, 16, 8192), seqs=seqs, tree=tree,
                **shape)


# ---------------------------------------------------------------- weights


def _gen(seed, key):
    h = seed
    for ch in key:
        h = (h * 1000003 + ord(ch)) % (1 << 61)
    return torch.Generator(device=DEV).manual_seed(h)


def _half_bytes(t):
    return t.to(torch.float16).contiguous().view(torch.uint8).reshape(*t.shape, 2)


class Weight:
    """rows x cols of one GGUF type: raw() its blocks, f64() its values."""

    def __init__(self, seed, key, dt, rows, cols, std=STD):
        self.dt, self.rows, self.cols = dt, rows, cols
        g = _gen(seed, key)

        def normal(*shape):
            return torch.randn(*shape, generator=g, device=DEV)

        def uniform(*shape):
            return torch.rand(*shape, generator=g, device=DEV)

        v = normal(rows, cols)
        if dt in (F16, F32):
            self.q = (v * std).to(torch.float16 if dt == F16 else torch.float32)
            return
        per = 256 if dt in (Q4_K, Q6_K) else 32
        nb = cols // per
        self.q = None
        if dt == Q4_0:
            self.d = (std / 2.8 * (0.9 + 0.2 * uniform(rows, nb))).to(torch.float16)
            self.q = (torch.round(v * 2.8) + 8).clamp(0, 15).to(torch.uint8)
        elif dt == Q8_0:
            self.d = (std / 42 * (0.9 + 0.2 * uniform(rows, nb))).to(torch.float16)
            self.q = torch.round(v * 42).clamp(-127, 127).to(torch.int8)
        elif dt == Q4_K:
            # d sc = one step of about 0.29 std, dmin m = 7.5 of them
            self.d = (std / 3.4 / 50 * (0.9 + 0.2 * uniform(rows, nb))).to(torch.float16)
            self.dmin = (std / 3.4 / 50 * 7.5 * (0.9 + 0.2 * uniform(rows, nb))).to(torch.float16)
            self.sc = (42 + 21 * uniform(rows, nb, 8)).to(torch.uint8)
            self.m = (42 + 21 * uniform(rows, nb, 8)).to(torch.uint8)
            self.q = torch.round(v * 3.4 + 7.5).clamp(0, 15).to(torch.uint8)
        elif dt == Q6_K:
            self.d = (std / 10 / 95 * (0.9 + 0.2 * uniform(rows, nb))).to(torch.float16)
            s = (64 + 63 * uniform(rows, nb, 16)).to(torch.int8)
            self.sc = torch.where(uniform(rows, nb, 16) < 0.5, s, -s)
            self.q = (torch.round(v * 10) + 32).clamp(0, 63).to(torch.uint8)
        self.nb = nb

    def raw(self):
        r, nb = self.rows, getattr(self, "nb", 0)
        if self.dt in (F16, F32):
            return self.q.contiguous().view(torch.uint8).reshape(-1)
        if self.dt == Q4_0:
            q = self.q.view(r, nb, 16, 2)
            parts = [_half_bytes(self.d), q[..., 0] | (q[..., 1] << 4)]
        elif self.dt == Q8_0:
            parts = [_half_bytes(self.d), self.q.view(torch.uint8).view(r, nb, 32)]
        elif self.dt == Q4_K:
            sc, m = self.sc, self.m
            s = torch.cat([sc[..., :4] | ((sc[..., 4:] >> 4) << 6), m[..., :4] | ((m[..., 4:] >> 4) << 6),
                           (sc[..., 4:] & 15) | ((m[..., 4:] & 15) << 4)], -1)
            q = self.q.view(r, nb, 4, 2, 32)
            parts = [_half_bytes(self.d), _half_bytes(self.dmin), s,
                     (q[..., 0, :] | (q[..., 1, :] << 4)).reshape(r, nb, 128)]
        else:
            q = self.q.view(r, nb, 2, 4, 32)
            lo, hi = q & 15, q >> 4
            ql = lo[..., :2, :] | (lo[..., 2:, :] << 4)
            qh = hi[..., 0, :] | (hi[..., 1, :] << 2) | (hi[..., 2, :] << 4) | (hi[..., 3, :] << 6)
            parts = [ql.reshape(r, nb, 128), qh.reshape(r, nb, 64), self.sc.view(torch.uint8),
                     _half_bytes(self.d)]
        return torch.cat(parts, -1).reshape(-1)

    def f64(self):
        r = self.rows
        if self.dt in (F16, F32):
            return self.q.double()
        nb, d = self.nb, self.d.double()
        if self.dt == Q4_0:
            w = d[..., None] * (self.q.view(r, nb, 32).double() - 8)
        elif self.dt == Q8_0:
            w = d[..., None] * self.q.view(r, nb, 32).double()
        elif self.dt == Q4_K:
            w = (d[..., None] * self.sc.double())[..., None] * self.q.view(r, nb, 8, 32).double()
            w = w - (self.dmin.double()[..., None] * self.m.double())[..., None]
        else:
            w = (d[..., None] * self.sc.double())[..., None] * (self.q.view(r, nb, 16, 16).double() - 32)
        return w.reshape(r, self.cols)


def _mix(mix, layer, layers, role):
    """The type of a model's tensor, as the file types choose them."""
    if mix == "q4_0":
        return F32 if role == "tok_embd" else Q4_0
    if mix == "q4_k_m":
        if role == "output":
            return Q6_K
        if role in ("v", "down"):
            more = layer < layers // 8 or layer >= 7 * layers // 8 or (layer - layers // 8) % 3 == 2
            return Q6_K if more else Q4_K
        return Q4_K
    if mix == "q8attn":
        return Q6_K if role == "output" else Q8_0 if role in ("q", "k", "v", "o") else Q4_K
    return TYPES[mix]


VARIANTS = 4  # layers share the weights of layer l % 4 where their types agree


def _layer_weights(case, seed, l):
    """name -> Weight of layer l's matrices."""
    d, hd, ff = case["d"], case["hd"], case["ff"]
    qd, kd = case["heads"] * hd, case["kv_heads"] * hd
    rows = dict(q=(qd, d), k=(kd, d), v=(kd, d), o=(d, qd))
    E = case.get("experts", 0)
    if E:
        rows.update(gate_inp=(E, d), gate_exps=(E * ff, d), up_exps=(E * ff, d),
                    down_exps=(E * ff, d))
    else:
        rows.update(gate=(ff, d), up=(ff, d), down=(ff, d))
    for role, (r, c) in rows.items():
        dt = F32 if role == "gate_inp" else _mix(case["mix"], l, case["layers"], role)
        key = "%d.%s.%d" % (l % VARIANTS, role, dt)
        yield role, key, dt, r, c, 2.0 / math.sqrt(d) if role == "gate_inp" else STD


def _norm(seed, key, d):
    return 1 + 0.1 * torch.randn(1, d, generator=_gen(seed, key), device=DEV)


# ---------------------------------------------------------------- programs' state

_context = None


def _ctx():
    global _context
    if _context is None:
        _context = ftx.Context(torch.cuda.current_device())
    return _context


class _Cache:
    """A KV cache that lives as long as whatever looks at its memory."""

    def __init__(self, kv):
        self.kv = kv

    def __del__(self):
        self.kv.free()


class _View:
    """Device memory of the library for torch to look at (a tensor made of
    it keeps it, and so `owner`, alive)."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(data=(ptr, False), shape=tuple(shape), strides=None,
                                             typestr=typestr, version=3)


class State:
    def __init__(self, case):
        self.case, self.held = case, []

    def hold(self, thing):
        self.held.append(thing)
        return thing

    def __del__(self):
        for thing in reversed(self.held):
            thing.free()
        self.held = []


def _upload(s, w, planes=1):
    raw = w.raw().cpu().numpy()
    ne = (w.cols, w.rows // planes, planes) if planes > 1 else (w.cols, w.rows)
    return s.hold(_ctx().upload(raw, w.dt, ne))


def _tree(case, rng):
    """parents of one sequence's draft nodes in breadth-first order, up to
    `tree` children each (0: a chain, None)."""
    if not case["tree"]:
        return None
    parents, level = [-1] * min(case["tree"], case["M"]), list(range(min(case["tree"], case["M"])))
    while len(parents) < case["M"]:
        nxt = []
        for p in level:
            for _ in range(int(rng.integers(1, case["tree"] + 1))):
                if len(parents) < case["M"]:
                    parents.append(p)
                    nxt.append(len(parents) - 1)
        level = nxt
    return np.array(parents, np.int32)


def _model_inputs(case, seed):
    """Tokens, parents and K / V context of every sequence."""
    rng = np.random.default_rng(seed)
    out = []
    for i in range(case.get("seqs", 1)):
        toks = rng.integers(0, case["vocab"], case["M"]).astype(np.int32)
        par = _tree(case, rng) if case["kind"] == "verify" else None
        g = _gen(seed, "kv%d" % i)
        kv = [torch.randn(case["layers"], case.get("ctx", 0), case["kv_heads"] * case["hd"], generator=g,
                          device=DEV).to(torch.float16) for _ in range(2)]
        out.append((toks, par, kv[0], kv[1]))
    return out


def _prepare_model(case, seed):
    s, ctx = State(case), _ctx()
    cfg = dict(n_layer=case["layers"], n_embd=case["d"], n_head=case["heads"],
               n_head_kv=case["kv_heads"], head_dim=case["hd"], n_ff=case["ff"],
               vocab=case["vocab"], rope_theta=case["theta"], n_expert=case.get("experts", 0),
               n_expert_used=case.get("used", 0))
    tensors, made = {}, {}
    for name in ("tok_embd", "output"):
        tensors[name] = _upload(s, Weight(seed, name, _mix(case["mix"], 0, 1, name), case["vocab"], case["d"]))
    norms = ["out_norm"] + ["blk.%d.%s" % (l, r) for l in range(case["layers"])
                            for r in ("attn_norm", "ffn_norm")]
    for name in norms:
        w = _norm(seed, name, case["d"])
        tensors[name] = s.hold(ctx.upload(w.cpu().numpy().view(np.uint8), F32, (case["d"], 1)))
    for l in range(case["layers"]):
        for role, key, dt, r, c, std in _layer_weights(case, seed, l):
            if key not in made:
                made[key] = _upload(s, Weight(seed, key, dt, r, c, std),
                                    case["experts"] if role.endswith("exps") else 1)
            tensors["blk.%d.%s" % (l, role)] = made[key]
    prefill = case["kind"] == "prefill"
    step = min(case["chunk"], case["M"]) if prefill else case["M"] * case["seqs"]
    s.model = s.hold(ctx.model(cfg, tensors, max_tokens=max(8, step)))
    past = 0 if prefill else case["ctx"]
    s.seqs = []
    for toks, par, k, v in _model_inputs(case, seed):
        kv = s.model.kv(past + case["M"] + 8)
        cache = _Cache(kv)
        kp, vp, _ = kv.pointers()
        L, cap, H, hd = case["layers"], kv.cap_alloc, case["kv_heads"], case["hd"]
        K = torch.as_tensor(_View(cache, kp, (L, cap, H * hd), "<f2"), device=DEV)
        V = torch.as_tensor(_View(cache, vp, (L, H, hd, cap), "<f2"), device=DEV)
        if past:
            K[:, :past] = k
            V[..., :past] = v.view(L, past, H, hd).permute(0, 2, 3, 1)
        kv.truncate(past)
        rows = min(case["chunk"], case["M"]) if prefill else case["M"]
        logits = torch.zeros(rows, case["vocab"], device=DEV)
        s.seqs.append((kv, toks, par, logits, K[:, past:past + case["M"]], V[..., past:past + case["M"]]))
    return s


def _draft(case, seed):
    """Target logits of the last committed token and of every draft node,
    draft distributions that resemble them, and tokens drawn from those."""
    M, V, T = case["M"], case["V"], case["temp"]
    g, rng = _gen(seed, "accept"), np.random.default_rng(seed)
    par = _tree(case, rng)
    parents = np.arange(-1, M - 1) if par is None else par
    rows = 3.0 * torch.randn(M + 1, V, generator=g, device=DEV)  # row 0: the base row
    q = torch.empty(M, V, device=DEV)
    props = torch.empty(M, dtype=torch.int64, device=DEV)
    dists = {}
    for i in range(M):
        p = int(parents[i])
        if p not in dists:  # children of one node share its draft distribution
            dists[p] = torch.softmax((rows[p + 1] + 0.7 * torch.randn(V, generator=g, device=DEV)) / T, 0)
        q[i] = dists[p]
        # inverse CDF of one uniform
        cdf = torch.cumsum(dists[p].double(), 0)
        u = torch.rand(1, generator=g, device=DEV, dtype=torch.float64) * cdf[-1]
        props[i] = torch.searchsorted(cdf, u).clamp(max=V - 1)[0]
    pd = q[torch.arange(M, device=DEV), props]
    return par, rows, q, props.cpu().numpy().astype(np.int32), pd.cpu().numpy()


def prepare(case, seed):
    if case["kind"] in ("verify", "prefill"):
        return _prepare_model(case, seed)
    s = State(case)
    if case["kind"] == "accept":
        s.parents, s.rows, s.q, s.props, s.pd = _draft(case, seed)
        s.rng = 1 + seed * 7919
        return s
    dt, M = TYPES[case["dt"]], case["M"]
    s.w = [_upload(s, w) for w in _op_weights(case, seed, dt)]
    s.x, s.y = _op_inputs(case, seed)
    if case["host"]:
        s.x, s.y = s.x.cpu().numpy(), s.y.cpu().numpy()
    return s


def _op_weights(case, seed, dt):
    if case["kind"] == "matmul":
        return [Weight(seed, "w", dt, case["N"], case["K"])]
    if case["kind"] == "down":
        return [Weight(seed, "w", dt, case["n_in"], case["N"])]
    return [Weight(seed, "w%d" % i, dt, case["IC"], case["K"]) for i in range(3)]


def _op_inputs(case, seed):
    """Activations: unit rows for a projection, SwiGLU outputs (small, with
    heavy tails) for the down form; the rows that the down and expert forms
    add to."""
    g = _gen(seed, "x")
    n = case["n_in"] if case["kind"] == "down" else case["K"]
    x = torch.randn(case["M"], n, generator=g, device=DEV)
    if case["kind"] == "down":
        x = torch.nn.functional.silu(x) * torch.randn(case["M"], n, generator=g, device=DEV)
    cols = case["K"] if case["kind"] == "expert" else case["N"]
    y = torch.zeros(case["M"], cols, device=DEV)
    return x, y


# ---------------------------------------------------------------- one pass


def run(s):
    case, ctx = s.case, _ctx()
    kind = case["kind"]
    if kind == "verify":
        if case["seqs"] == 1:
            kv, toks, par, logits, K, V = s.seqs[0]
            kv.truncate(case["ctx"])
            if case["M"] == 1:
                s.model.step(kv, int(toks[0]), logits.data_ptr())
            else:
                s.model.verify(kv, toks, logits.data_ptr(), parents=par)
        else:
            for q in s.seqs:
                q[0].truncate(case["ctx"])
            s.model.verify_batch([(q[0], q[1], q[3].data_ptr(), q[2], False) for q in s.seqs])
        return [{"logits": q[3], "k": q[4], "v": q[5]} for q in s.seqs]
    if kind == "prefill":
        kv, toks, _, logits, K, V = s.seqs[0]
        kv.truncate(0)
        n = s.model.prefill(kv, toks, logits.data_ptr(), chunk=case["chunk"])
        return {"logits": logits[:n], "k": K, "v": V}
    if kind == "accept":
        M, V = case["M"], case["V"]
        if case["tree"]:
            r = ctx.accept(s.rows.data_ptr(), s.rows[1:].data_ptr(), M, V, s.props, ftx.ACCEPT_RESIDUAL,
                           temp=case["temp"], rng=s.rng, parents=s.parents, q_ptr=s.q.data_ptr())
        else:
            r = ctx.accept(s.rows.data_ptr(), s.rows[1:].data_ptr(), M, V, s.props, ftx.ACCEPT_RATIO,
                           temp=case["temp"], rng=s.rng, pd=s.pd)
        path = r["accepted"] + [-1] * (M - len(r["accepted"]))
        words = [w for n in ("rng", "sampler_state") for w in (r[n] >> 32, r[n] & 0xFFFFFFFF)]
        return {"path": np.array(path), "bonus": r["bonus"], "states": np.array(words, np.int64),
                "margin": np.array([r["margin"]], np.float32)}
    M, lib = case["M"], ctx.lib
    x, y = (s.x.ctypes.data, s.y.ctypes.data) if case["host"] else (s.x.data_ptr(), s.y.data_ptr())
    if kind == "matmul":
        ctx.check(lib.ftx_matmul(ctx.h, x, M, case["K"], s.w[0].handle, y))
        return s.y
    # the down and expert forms add to y: a layer starts from its own rows
    if case["host"]:
        s.y.fill(0)
    else:
        s.y.zero_()
    if kind == "down":
        ctx.check(lib.ftx_down_axpy(ctx.h, x, M, case["n_in"], s.w[0].handle, y))
    else:
        strides = [t.nbytes // case["IC"] for t in s.w]
        job = ftx.ExpertJob(x, y, s.w[0].ptr, s.w[1].ptr, s.w[2].ptr, TYPES[case["dt"]], 0, M,
                            case["K"], case["IC"], strides[0], strides[2])
        ctx.check(lib.ftx_expert_chunk(ctx.h, job))
    return s.y


# ---------------------------------------------------------------- what a pass cannot do without


def _row_bytes(dt, cols):
    return ftx.row_bytes(dt, cols)


def work(case):
    kind = case["kind"]
    if kind == "accept":
        # every target row once; the draft rows only where a child is rejected
        return dict(bytes=4.0 * (case["M"] + 1) * case["V"], flops=4.0 * (case["M"] + 1) * case["V"])
    if kind in ("matmul", "down", "expert"):
        dt = TYPES[case["dt"]]
        if kind == "matmul":
            n, act = case["N"] * _row_bytes(dt, case["K"]), case["K"] + case["N"]
            mac = case["N"] * case["K"]
        elif kind == "down":
            n, act = case["n_in"] * _row_bytes(dt, case["N"]), case["n_in"] + 2 * case["N"]
            mac = case["n_in"] * case["N"]
        else:
            n, act = 3 * case["IC"] * _row_bytes(dt, case["K"]), 3 * case["K"]
            mac = 3 * case["IC"] * case["K"]
        return dict(bytes=float(n + 4 * case["M"] * act), flops=2.0 * case["M"] * mac)
    M, seqs = case["M"], case.get("seqs", 1)
    tokens, past = M * seqs, case.get("ctx", 0)
    E, U = case.get("experts", 0), case.get("used", 0)
    nbytes = flops = 0.0
    for l in range(case["layers"]):
        for role, key, dt, r, c, std in _layer_weights(case, 0, l):
            share = min(E, tokens * U) / E if role.endswith("exps") else 1.0
            nbytes += share * r * _row_bytes(dt, c)
            flops += 2.0 * tokens * r * c * (U / E if role.endswith("exps") else 1.0)
        keys = past + M if kind == "verify" else M / 2
        nbytes += seqs * 2.0 * (past + M) * case["kv_heads"] * case["hd"] * 2
        flops += 4.0 * tokens * keys * case["heads"] * case["hd"]
    rows = tokens if kind == "verify" else (M - 1) % case["chunk"] + 1
    nbytes += case["vocab"] * _row_bytes(_mix(case["mix"], 0, 1, "output"), case["d"])
    nbytes += 4.0 * rows * case["vocab"] + tokens * _row_bytes(_mix(case["mix"], 0, 1, "tok_embd"), case["d"])
    flops += 2.0 * rows * case["vocab"] * case["d"]
    return dict(bytes=nbytes, flops=flops)


def tolerance(case):
    """About four times the error against exact() that the paths show."""
    kind = case["kind"]
    if kind == "accept":
        return {"rel": 1e-5}  # the decision margin; tokens and states are whole numbers
    if kind in ("matmul", "down", "expert"):
        # 32-bit sums (1e-7 to 6e-7 seen); up to 8 rows of the K types'
        # projections go through activations of two int8 limbs
        limbs = kind == "matmul" and case["M"] <= 8 and case["dt"] in ("q4_k", "q6_k")
        return {"rel": 2e-4 if limbs else 1e-5}
    if case["mix"] in ("q4_0", "q8_0", "f16"):
        return {"rel": 1.5e-4}  # fp16 rounding of the K / V rows: 3e-5 seen
    # the int8 limbs of the K types: 2.3e-4 after 4 layers, 1.8e-3 after 32
    return {"rel": 7e-3 if case["layers"] > 8 else 1e-3}


# ---------------------------------------------------------------- 64 bits


def _exact_model(case, seed):
    L, d, H, KH, hd = case["layers"], case["d"], case["heads"], case["kv_heads"], case["hd"]
    ins = _model_inputs(case, seed)
    past = case.get("ctx", 0)
    half = hd // 2
    freq = torch.tensor([case["theta"] ** (-2.0 * p / hd) for p in range(half)], dtype=torch.float64,
                        device=DEV)
    embd = Weight(seed, "tok_embd", _mix(case["mix"], 0, 1, "tok_embd"), case["vocab"], d).f64()
    toks = torch.from_numpy(np.concatenate([i[0] for i in ins]).astype(np.int64)).to(DEV)
    x = embd[toks]
    del embd
    M = case["M"]
    depth, mask = [], []
    for t, par, k, v in ins:
        par = np.arange(-1, M - 1) if par is None else par
        dep = np.zeros(M, np.int64)
        see = np.zeros((M, M), bool)
        for i in range(M):
            if par[i] >= 0:
                dep[i] = dep[par[i]] + 1
                see[i] = see[par[i]]
            see[i, i] = True
        depth.append(dep)
        mask.append(torch.from_numpy(np.concatenate([np.ones((M, past), bool), see], 1)).to(DEV))
    pos = past + torch.from_numpy(np.concatenate(depth)).to(DEV).double()
    cos, sin = torch.cos(pos[:, None] * freq), torch.sin(pos[:, None] * freq)

    def rms(t, w):
        return t / torch.sqrt((t * t).mean(-1, keepdim=True) + float(np.float32(1e-5))) * w.double()

    def rope(t, n):
        t = t.view(-1, n, half, 2)
        c, s = cos[:, None], sin[:, None]
        return torch.stack([t[..., 0] * c - t[..., 1] * s, t[..., 0] * s + t[..., 1] * c], -1).reshape(-1, n, hd)

    ks, vs = [[] for _ in ins], [[] for _ in ins]
    for l in range(L):
        ws = {}
        for role, key, dt, r, c, std in _layer_weights(case, seed, l):
            ws[role] = Weight(seed, key, dt, r, c, std)
        xn = rms(x, _norm(seed, "blk.%d.attn_norm" % l, d))
        q = rope(xn @ ws["q"].f64().T, H)
        k = rope(xn @ ws["k"].f64().T, KH)
        v = (xn @ ws["v"].f64().T).view(-1, KH, hd)
        att = []
        for i, (t, par, kc, vc) in enumerate(ins):
            sl = slice(i * M, (i + 1) * M)
            ks[i].append(k[sl].reshape(M, KH * hd))
            vs[i].append(v[sl].permute(1, 2, 0))
            # the cache holds halves, and attention reads the cache
            keys = torch.cat([kc[l].view(past, KH, hd), k[sl].half()], 0).double()
            vals = torch.cat([vc[l].view(past, KH, hd), v[sl].half()], 0).double()
            heads = []
            for h in range(H):
                sc = q[sl, h] @ keys[:, h // (H // KH)].T / math.sqrt(hd)
                p = torch.softmax(sc.masked_fill(~mask[i], -math.inf), -1)
                heads.append(p @ vals[:, h // (H // KH)])
            att.append(torch.stack(heads, 1).reshape(M, H * hd))
        x = x + torch.cat(att, 0) @ ws["o"].f64().T
        xn = rms(x, _norm(seed, "blk.%d.ffn_norm" % l, d))
        if not case.get("experts", 0):
            h = torch.nn.functional.silu(xn @ ws["gate"].f64().T) * (xn @ ws["up"].f64().T)
            x = x + h @ ws["down"].f64()
            continue
        ff = case["ff"]
        p = torch.softmax(xn @ ws["gate_inp"].f64().T, -1)
        top, idx = torch.topk(p, case["used"], -1)
        top = top / top.sum(-1, keepdim=True)
        add = torch.zeros_like(x)
        for e in range(case["experts"]):
            part = {}
            for role in ("gate_exps", "up_exps", "down_exps"):
                w = ws[role]
                one = object.__new__(Weight)
                one.__dict__.update(w.__dict__)
                one.rows = ff
                for name in ("q", "d", "dmin", "sc", "m"):
                    if hasattr(w, name):
                        setattr(one, name, getattr(w, name)[e * ff:(e + 1) * ff])
                part[role] = one.f64()
            h = torch.nn.functional.silu(xn @ part["gate_exps"].T) * (xn @ part["up_exps"].T)
            wt = (top * (idx == e)).sum(-1, keepdim=True)
            add += wt * (h @ part["down_exps"])
        x = x + add
    xn = rms(x, _norm(seed, "out_norm", d))
    if case["kind"] == "prefill":
        xn = xn[(M - 1) // case["chunk"] * case["chunk"]:]
    logits = xn @ Weight(seed, "output", _mix(case["mix"], 0, 1, "output"), case["vocab"], d).f64().T
    if case["kind"] == "prefill":
        return {"logits": logits, "k": torch.stack(ks[0]), "v": torch.stack(vs[0])}
    return [{"logits": logits[i * M:(i + 1) * M], "k": torch.stack(ks[i]), "v": torch.stack(vs[i])}
            for i in range(len(ins))]


def exact(case, seed):
    kind = case["kind"]
    if kind == "accept":
        return None
    if kind in ("verify", "prefill"):
        return _exact_model(case, seed)
    x, y = _op_inputs(case, seed)
    w = [t.f64() for t in _op_weights(case, seed, TYPES[case["dt"]])]
    x = x.double()
    if kind == "matmul":
        return x @ w[0].T
    if kind == "down":
        return x @ w[0]
    return (torch.nn.functional.silu(x @ w[0].T) * (x @ w[1].T)) @ w[2]
