"""The work this framework is used for, as cases that a program can time and check.

`listed()` names them, `draw(rng)` gives more of the same ranges, `prepare` makes what a program
holds before the call, `run` is one pass through the public entry points, `work` what the pass
cannot do without, `exact` its result in 64 bits by plain torch, and `tolerance` how far another
correct implementation at the same precision may be from it.

Shapes are those of the repository's model (Llama-3.2-1B: hidden 2048, 32 query and 8 KV heads of
64, MLP width 8192, vocabulary 128256, 16 layers, KV pages of 16 positions) and, for the single
operators, generic widths around it.
"""
from __future__ import annotations

import importlib
import math

import numpy as np
import torch

from __graft_entry__ import load_llmk

llmk = load_llmk()
weights = importlib.import_module("llmk.weights")

DEV = "cuda"
PAGE, HEAD, EPS = 16, 64, 1e-5
HIDDEN, HEADS, KV_HEADS, INTER, VOCAB, LAYERS = 2048, 32, 8, 8192, 128256, 16
QDIM, KVDIM = HEADS * HEAD, KV_HEADS * HEAD
ROPE = (500000.0, 32.0, 1.0, 4.0, 8192.0)  # theta, factor, low, high, original max position
BLOCK_LAYERS, BLOCK_VOCAB = 2, 8192  # the decoder-block cases: two layers and a small head


def listed():
    return [
        # The smallest call: the norm between two projections of a 16-sequence decode step, where
        # the launch and the host path are all there is.
        dict(name="add_rmsnorm_16", kind="add_rmsnorm", rows=16, hidden=HIDDEN),
        # The same over a prefill of 8192 tokens: a stream over HBM.
        dict(name="add_rmsnorm_8192", kind="add_rmsnorm", rows=8192, hidden=HIDDEN),
        # The MLP's activation over a prefill of 8192 tokens.
        dict(name="swiglu_8192", kind="swiglu", n=8192 * INTER),
        # Everything of a decode step but its projections and attention, for callers that bring
        # their own GEMMs: 256 sequences, 16 layers.
        dict(name="nongemm_pass_256", kind="nongemm_pass", seqs=256, layers=LAYERS, norms=1,
             max_len=2048),
        # Decode attention of a full batch at the context lengths of a serving mix ...
        dict(name="attention_256", kind="attention", seqs=256, max_len=2048),
        # ... and of a few sequences with long contexts.
        dict(name="attention_5_long", kind="attention", seqs=5, max_len=16384),
        # The MLP of one sequence's decode step: weights streamed for one row.
        dict(name="mlp_1", kind="mlp", rows=1, hidden=HIDDEN, inter=INTER),
        # The MLP of a mid-size batch, through the projections that any caller can use.
        dict(name="mlp_40", kind="mlp", rows=40, hidden=HIDDEN, inter=INTER),
        # Decoder layers in the engine: a decode step of 64 sequences ...
        dict(name="block_decode_64", kind="block", seqs=64, max_len=2048, prompt=0, start=0),
        # ... and the prefill of one prompt of odd length.
        dict(name="block_prefill_1507", kind="block", seqs=0, max_len=1, prompt=1507, start=0),
        # Whole decode steps, the embedding, 16 layers and the head: a small batch, where latency
        # counts, and a full one.
        dict(name="step_8", kind="step", seqs=8, max_len=2048),
        dict(name="step_256", kind="step", seqs=256, max_len=2048),
    ]


def _log_int(rng, lo, hi):
    """A whole number in [lo, hi], uniform over its logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))
    return min(hi, max(lo, int(v)))


def draw(rng):
    kind = rng.choice(["add_rmsnorm", "swiglu", "nongemm_pass", "attention", "attention", "mlp",
                       "mlp", "block", "block", "block", "step"])
    if kind == "add_rmsnorm":
        return dict(kind=kind, rows=_log_int(rng, 1, 8192),
                    hidden=rng.choice([1024, 1608, HIDDEN, 3072, 4096]))
    if kind == "swiglu":
        return dict(kind=kind, n=_log_int(rng, INTER, 8192 * INTER))
    if kind == "nongemm_pass":
        return dict(kind=kind, seqs=_log_int(rng, 1, 256), layers=rng.randint(1, LAYERS),
                    norms=rng.choice([1, 2]), max_len=rng.randint(16, 2048))
    if kind == "attention":
        seqs = _log_int(rng, 1, 256)
        return dict(kind=kind, seqs=seqs, max_len=_log_int(rng, 48, min(16384, 524288 // seqs)))
    if kind == "mlp":
        hidden = rng.choice([1024, HIDDEN, HIDDEN, 4096])
        return dict(kind=kind, rows=_log_int(rng, 1, 2048), hidden=hidden,
                    inter=hidden * rng.choice([3, 4]))
    if kind == "block":
        # decode steps, prompts (some behind a cached prefix), and passes that mix the two
        what = rng.choice(["decode", "decode", "prompt", "prompt", "mixed"])
        seqs = 0 if what == "prompt" else _log_int(rng, 1, 256 if what == "decode" else 32)
        prompt = 0 if what == "decode" else _log_int(rng, 9, 2048 if what == "prompt" else 512)
        start = rng.choice([0, 0, rng.randint(1, 1024)]) if prompt else 0
        return dict(kind=kind, seqs=seqs, max_len=rng.randint(32, 2048) if seqs else 1,
                    prompt=prompt, start=start)
    return dict(kind="step", seqs=_log_int(rng, 1, 256), max_len=rng.randint(32, 2048))


# ---------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _normal(shape, g, mean=0.0, std=1.0):
    t = torch.randn(shape, generator=g, device=DEV, dtype=torch.float32)
    return t.mul_(std).add_(mean).half()


def _ints(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.int32)).to(DEV)


def _inv_freq():
    return torch.tensor(llmk.compute_rope_inv_freq(HEAD, *ROPE), dtype=torch.float32, device=DEV)


def _pages(lens, rng):
    """(block tables [n, widest], pages in all) for sequences of these lengths, the pages given
    out in a shuffled order as a running server's free list does."""
    need = [(int(n) + PAGE - 1) // PAGE for n in lens]
    order = rng.permutation(sum(need)).astype(np.int32)
    tables = np.zeros((len(need), max(need)), np.int32)
    at = 0
    for b, k in enumerate(need):
        tables[b, :k] = order[at:at + k]
        at += k
    return tables, sum(need)


def _lens(case):
    """Context lengths of the case's sequences: fixed by the case, so that its work is, uniform
    in [1, max_len] with the longest one present."""
    r = np.random.default_rng([case["seqs"], case["max_len"]])
    lens = r.integers(1, case["max_len"] + 1, case["seqs"])
    if lens.size:
        lens[r.integers(0, lens.size)] = case["max_len"]
    return lens


class _Row:
    """The rows of one engine pass: a decode row per sequence, then the prompt's rows."""

    def __init__(self, case, seed):
        rng = np.random.default_rng(seed)
        vocab = BLOCK_VOCAB if case["kind"] == "block" else VOCAB
        lens = _lens(case)
        prompt, start = case.get("prompt", 0), case.get("start", 0)
        every = np.concatenate([lens, [prompt + start]]) if prompt else lens
        tables, self.num_pages = _pages(every, rng)
        self.decode, self.prompt, self.start, self.lens = lens.size, prompt, start, lens
        self.seq_tables = tables
        self.positions = np.concatenate([lens - 1, start + np.arange(prompt)]).astype(np.int32)
        self.tables = np.concatenate([tables[:lens.size],
                                      np.repeat(tables[-1:], prompt, 0)]).astype(np.int32)
        self.n = self.positions.size
        self.tokens = rng.integers(0, vocab, self.n).astype(np.int32)
        # logits of every decode row and of the prompt's last row
        self.logit_rows = (np.concatenate([np.arange(lens.size), [self.n - 1]]).astype(np.int32)
                           if prompt else None)


def _model(case):
    if case["kind"] == "block":
        return llmk.ModelConfig(n_layers=BLOCK_LAYERS, vocab=BLOCK_VOCAB)
    return llmk.ModelConfig()


def _model_weights(case, seed):
    return weights.random_weights(_model(case), seed, device=DEV)


def _fill(case, rows, layer, seed):
    """The cached keys and values of one layer before the pass."""
    g = _gen(seed * 64 + layer + 1)
    n = rows.num_pages * PAGE * KVDIM
    return _normal((n,), g), _normal((n,), g)


class _Buffer:
    """An engine buffer as torch sees it; keeps its engine alive."""

    def __init__(self, engine, ptr, shape):
        self.engine = engine
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr="<f2", version=3,
                                             data=(ptr, False), strides=None)


def _view(engine, which, layer, shape):
    return torch.as_tensor(_Buffer(engine, engine.buffer_ptr(which, layer), shape), device=DEV)


_stream = None


def _engine_stream():
    """The stream a serving loop drives its engines on."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream


# ---------------------------------------------------------------------------------------------
# prepare
# ---------------------------------------------------------------------------------------------
def prepare(case, seed):
    return _KINDS[case["kind"]].prepare(case, seed)


def run(state):
    return state["kind"].run(state)


def work(case):
    return _KINDS[case["kind"]].work(case)


def exact(case, seed):
    return _KINDS[case["kind"]].exact(case, seed)


def tolerance(case):
    return _KINDS[case["kind"]].tolerance(case)


def _rmsnorm64(x, w):
    x = x.double()
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _swiglu64(g, u):
    return torch.nn.functional.silu(g.double()) * u.double()


def _rope64(x, positions, inv_freq):
    """x [n, heads, 64]; positions [n]."""
    a = positions.double()[:, None] * inv_freq.double()[None, :]
    c, s = torch.cos(a)[:, None, :], torch.sin(a)[:, None, :]
    lo, hi = x.double().chunk(2, -1)
    return torch.cat([lo * c - hi * s, hi * c + lo * s], -1)


def _attend64(q, k, v, mask=None):
    """q [m, heads, 64] over k, v [s, kv heads, 64]; mask [m, s] of the positions left out."""
    m = q.shape[0]
    g = q.shape[1] // k.shape[1]
    qg = q.double().view(m, k.shape[1], g, HEAD).permute(1, 2, 0, 3).reshape(k.shape[1], g * m, HEAD)
    kt, vt = k.double().permute(1, 0, 2), v.double().permute(1, 0, 2)
    s = torch.matmul(qg, kt.transpose(1, 2).contiguous()) / math.sqrt(HEAD)
    if mask is not None:
        s.masked_fill_(mask.repeat(g, 1)[None], float("-inf"))
    o = torch.matmul(torch.softmax(s, -1), vt.contiguous())
    return o.view(k.shape[1], g, m, HEAD).permute(2, 0, 1, 3).reshape(m, -1, HEAD)


class _AddRmsnorm:
    """residual += x, out = rmsnorm(residual)."""

    @staticmethod
    def inputs(case, seed):
        g = _gen(seed)
        shape = (case["rows"], case["hidden"])
        return _normal(shape, g), _normal(shape, g), _normal((case["hidden"],), g, 1.0, 0.1)

    @classmethod
    def prepare(cls, case, seed):
        residual, x, w = cls.inputs(case, seed)
        return dict(kind=cls, residual=residual, x=x, w=w, out=torch.empty_like(x), **{
            k: case[k] for k in ("rows", "hidden")})

    @staticmethod
    def run(s):
        llmk.add_rmsnorm(s["residual"], s["x"], s["w"], s["out"], s["rows"], s["hidden"], EPS)
        return s["residual"], s["out"]

    @staticmethod
    def work(case):
        n = case["rows"] * case["hidden"]
        return dict(bytes=4 * n * 2 + case["hidden"] * 2, flops=5 * n)

    @classmethod
    def exact(cls, case, seed):
        residual, x, w = cls.inputs(case, seed)
        r = residual.double() + x.double()
        return r, _rmsnorm64(r, w)

    @staticmethod
    def tolerance(case):
        return {"rel": 1.4e-3, "max": 5e-3}


class _Swiglu:
    """out = silu(gate) * up."""

    @staticmethod
    def inputs(case, seed):
        g = _gen(seed)
        return _normal((case["n"],), g), _normal((case["n"],), g)

    @classmethod
    def prepare(cls, case, seed):
        gate, up = cls.inputs(case, seed)
        return dict(kind=cls, gate=gate, up=up, out=torch.empty_like(gate), n=case["n"])

    @staticmethod
    def run(s):
        llmk.swiglu(s["gate"], s["up"], s["out"], s["n"])
        return s["out"]

    @staticmethod
    def work(case):
        return dict(bytes=3 * case["n"] * 2, flops=5 * case["n"])

    @classmethod
    def exact(cls, case, seed):
        return _swiglu64(*cls.inputs(case, seed))

    @staticmethod
    def tolerance(case):
        return {"rel": 1.2e-3, "max": 5e-3}


class _NongemmPass:
    """A decode step's embedding, norms, RoPE + K/V scatter and SwiGLU over all layers."""

    @staticmethod
    def inputs(case, seed):
        g, rng = _gen(seed), np.random.default_rng(seed)
        n, lens = case["seqs"], _lens(case)
        tables, pages = _pages(lens, rng)
        table = _normal((VOCAB, HIDDEN), g, 0.0, 0.02)
        lay, norms = case["layers"], case["norms"]
        # one tensor per operand, layer by layer along its first axis
        a = dict(x=_normal((lay, n, HIDDEN), g), norm_w=_normal((lay, HIDDEN), g, 1.0, 0.1),
                 q=_normal((lay, n, HEADS, HEAD), g), k=_normal((lay, n, KV_HEADS, HEAD), g),
                 v=_normal((lay, n, KV_HEADS, HEAD), g), gate=_normal((lay, n, INTER), g),
                 up=_normal((lay, n, INTER), g))
        for pool in ("k_pool", "v_pool"):
            a[pool] = torch.empty((lay, pages * PAGE, KVDIM), dtype=torch.float16, device=DEV)
            for l in range(lay):
                a[pool][l] = _normal((pages * PAGE, KVDIM), g)
        if norms == 2:
            a.update(x2=_normal((lay, n, HIDDEN), g), norm_w2=_normal((lay, HIDDEN), g, 1.0, 0.1))
        return dict(table=table, ids=_ints(rng.integers(0, VOCAB, n)), tables=_ints(tables),
                    positions=_ints(lens - 1), layers=a, max_pages=tables.shape[1])

    @classmethod
    def prepare(cls, case, seed):
        inp = cls.inputs(case, seed)
        n, a = case["seqs"], inp["layers"]
        a.update(normed=torch.empty_like(a["x"]), act=torch.empty_like(a["gate"]))
        if "x2" in a:
            a["normed2"] = torch.empty_like(a["x2"])
        residual = torch.empty((n, HIDDEN), dtype=torch.float16, device=DEV)
        p = llmk.DecodeNonGemmPass(inp["table"], inp["ids"], residual, inp["tables"],
                                   inp["positions"], _inv_freq(),
                                   [{k: t[l] for k, t in a.items()} for l in range(case["layers"])],
                                   n_heads=HEADS, n_kv_heads=KV_HEADS, head_dim=HEAD, inter=INTER,
                                   page_size=PAGE, max_pages=inp["max_pages"], eps=EPS)
        names = ("q", "k_pool", "v_pool", "normed", "act") + (("normed2",) if "x2" in a else ())
        return dict(kind=cls, plan=p, out=dict(residual=residual, **{k: a[k] for k in names}))

    @staticmethod
    def run(s):
        s["plan"].run_fused()
        return s["out"]

    @staticmethod
    def work(case):
        n, lay, norms = case["seqs"], case["layers"], case["norms"]
        row = n * HIDDEN * 2
        per = (norms * (2 * row + HIDDEN * 2) + 2 * n * QDIM * 2 + 4 * n * KVDIM * 2
               + 3 * n * INTER * 2)
        return dict(bytes=2 * row + lay * per, flops=lay * n * (5 * norms * HIDDEN + 5 * INTER
                                                                + 6 * (QDIM + KVDIM)))

    @classmethod
    def exact(cls, case, seed):
        inp = cls.inputs(case, seed)
        inv, pos, a = _inv_freq(), inp["positions"], inp["layers"]
        n = case["seqs"]
        r = inp["table"][inp["ids"].long()].double()
        out = dict(q=torch.stack([_rope64(q, pos, inv) for q in a["q"]]),
                   act=_swiglu64(a["gate"], a["up"]), k_pool=a["k_pool"].double(),
                   v_pool=a["v_pool"].double())
        page = inp["tables"].long().gather(1, (pos.long() // PAGE)[:, None])[:, 0]
        at = page * PAGE + pos % PAGE
        normed, normed2 = [], []
        for l in range(case["layers"]):
            r = r + a["x"][l].double()
            normed.append(_rmsnorm64(r, a["norm_w"][l]))
            if "x2" in a:
                r = r + a["x2"][l].double()
                normed2.append(_rmsnorm64(r, a["norm_w2"][l]))
            out["k_pool"][l, at] = _rope64(a["k"][l], pos, inv).view(n, KVDIM)
            out["v_pool"][l, at] = a["v"][l].double().view(n, KVDIM)
        out.update(residual=r, normed=torch.stack(normed))
        if normed2:
            out["normed2"] = torch.stack(normed2)
        return out

    @staticmethod
    def tolerance(case):
        return {"rel": 2.5e-3, "max": 2e-2}


class _Attention:
    """Split-KV decode attention over the paged pool, one query token per sequence."""

    @staticmethod
    def inputs(case, seed):
        g, rng = _gen(seed), np.random.default_rng(seed)
        lens = _lens(case)
        tables, pages = _pages(lens, rng)
        return dict(q=_normal((lens.size, HEADS, HEAD), g), k_pool=_normal((pages * PAGE, KVDIM), g),
                    v_pool=_normal((pages * PAGE, KVDIM), g), tables=_ints(tables),
                    lens=_ints(lens), host_lens=lens, max_pages=tables.shape[1])

    @classmethod
    def prepare(cls, case, seed):
        a = cls.inputs(case, seed)
        n = case["seqs"]
        splits = llmk.choose_num_splits(n, KV_HEADS, case["max_len"])
        ws = torch.empty(max(1, llmk.attention_decode_fast_workspace_floats(n, HEADS, splits)),
                         dtype=torch.float32, device=DEV)
        return dict(kind=cls, n=n, splits=splits, ws=ws, out=torch.empty_like(a["q"]), **a)

    @staticmethod
    def run(s):
        llmk.attention_decode_fast(s["q"], s["k_pool"], s["v_pool"], s["tables"], s["lens"],
                                   s["out"], s["ws"], s["n"], s["max_pages"], PAGE, HEADS,
                                   KV_HEADS, HEAD, s["splits"])
        return s["out"]

    @staticmethod
    def work(case):
        total, n = int(_lens(case).sum()), case["seqs"]
        return dict(bytes=total * 2 * KVDIM * 2 + 2 * n * QDIM * 2, flops=4 * total * QDIM)

    @classmethod
    def exact(cls, case, seed):
        a = cls.inputs(case, seed)
        out = []
        for b, n in enumerate(a["host_lens"]):
            i = torch.arange(int(n), device=DEV)
            rows = a["tables"][b].long()[i // PAGE] * PAGE + i % PAGE
            out.append(_attend64(a["q"][b:b + 1], a["k_pool"][rows].view(-1, KV_HEADS, HEAD),
                                 a["v_pool"][rows].view(-1, KV_HEADS, HEAD)))
        return torch.cat(out)

    @staticmethod
    def tolerance(case):
        return {"rel": 1e-3, "max": 1e-2}


class _Mlp:
    """residual += down(swiglu(gate_up(rmsnorm(residual)))): the MLP half of a layer, through the
    fused few-rows projections up to 8 rows and the general ones beyond."""

    @staticmethod
    def inputs(case, seed):
        g = _gen(seed)
        t, h, i = case["rows"], case["hidden"], case["inter"]
        return dict(residual=_normal((t, h), g), x=_normal((t, h), g),
                    norm_w=_normal((h,), g, 1.0, 0.1), w_gu=_normal((2 * i, h), g, 0.0, 0.02),
                    w_down=_normal((h, i), g, 0.0, 0.02))

    @classmethod
    def prepare(cls, case, seed):
        a = cls.inputs(case, seed)
        t, h, i = case["rows"], case["hidden"], case["inter"]
        half = dict(dtype=torch.float16, device=DEV)
        return dict(kind=cls, t=t, h=h, i=i, blas=llmk.Blas(), normed=torch.empty((t, h), **half),
                    gu=torch.empty((t, 2 * i), **half), act=torch.empty((t, i), **half),
                    y=torch.empty((t, h), **half), **a)

    @staticmethod
    def run(s):
        t, h, i = s["t"], s["h"], s["i"]
        if t <= llmk.LINEAR_ROWS_MAX:
            llmk.linear_rows_swiglu(s["residual"], s["norm_w"], EPS, s["w_gu"], s["act"], t, h, i)
            llmk.linear_rows_residual(s["act"], s["w_down"], s["residual"], t, i, h)
            return s["act"], s["residual"]
        llmk.add_rmsnorm(s["residual"], s["x"], s["norm_w"], s["normed"], t, h, EPS)
        llmk.linear(s["blas"], s["normed"], s["w_gu"], s["gu"], t, h, 2 * i)
        llmk.swiglu_rows(s["gu"], s["act"], t, i)
        llmk.linear(s["blas"], s["act"], s["w_down"], s["y"], t, i, h)
        return s["residual"], s["normed"], s["act"], s["y"]

    @staticmethod
    def work(case):
        t, h, i = case["rows"], case["hidden"], case["inter"]
        return dict(bytes=3 * h * i * 2 + 4 * t * h * 2, flops=6 * t * h * i)

    @classmethod
    def exact(cls, case, seed):
        a = cls.inputs(case, seed)
        t, i = case["rows"], case["inter"]
        few = t <= llmk.LINEAR_ROWS_MAX
        r = a["residual"].double()
        if not few:
            r = r + a["x"].double()
        normed = _rmsnorm64(r, a["norm_w"])
        gu = normed @ a["w_gu"].double().t()
        act = _swiglu64(gu[:, :i], gu[:, i:])
        y = act @ a["w_down"].double().t()
        return (act, r + y) if few else (r, normed, act, y)

    @staticmethod
    def tolerance(case):
        return {"rel": 3e-3, "max": 3e-2}


class _Forward:
    """One engine pass: rows uploaded, embedding, layers, head. Decode steps go through the
    engine's graph cache, passes with a prompt are enqueued directly, as the scheduler does."""

    @classmethod
    def prepare(cls, case, seed):
        rows = _Row(case, seed)
        cfg = _model(case)
        e = llmk.Engine(cfg, max_rows=rows.n, max_pages=rows.tables.shape[1],
                        num_pages=rows.num_pages)
        e.set_weights(*weights.engine_layers(_model_weights(case, seed), cfg))
        for l in range(cfg.n_layers):
            k, v = _fill(case, rows, l, seed)
            e.write_pool(llmk.BUF_K_POOL, l, k)
            e.write_pool(llmk.BUF_V_POOL, l, v)
        nl = rows.n if rows.logit_rows is None else rows.logit_rows.size
        out = dict(logits=_view(e, llmk.BUF_LOGITS, 0, (nl, cfg.vocab)),
                   residual=_view(e, llmk.BUF_RESIDUAL, 0, (rows.n, cfg.hidden)))
        if case["kind"] == "block":
            shape = (rows.num_pages * PAGE, KVDIM)
            for name, which in (("k_pool", llmk.BUF_K_POOL), ("v_pool", llmk.BUF_V_POOL)):
                out[name] = [_view(e, which, l, shape) for l in range(cfg.n_layers)]
        return dict(kind=cls, engine=e, rows=rows, out=out, stream=_engine_stream())

    @staticmethod
    def run(s):
        e, r, st = s["engine"], s["rows"], s["stream"]
        e.set_rows(r.tokens, r.positions, r.tables, r.logit_rows, stream=st)
        if r.logit_rows is None:
            e.forward_graph(r.n, stream=st)
        else:
            e.forward(r.n, r.logit_rows.size, stream=st)
        return s["out"]

    @staticmethod
    def work(case):
        lens, prompt, start = _lens(case), case.get("prompt", 0), case.get("start", 0)
        block = case["kind"] == "block"
        layers, vocab = (BLOCK_LAYERS, BLOCK_VOCAB) if block else (LAYERS, VOCAB)
        n, nl = lens.size + prompt, lens.size + (1 if prompt else 0)
        mats = HIDDEN * (2 * QDIM + 2 * KVDIM + 3 * INTER)
        cached = int(lens.sum()) + (prompt + start if prompt else 0)
        pairs = int(lens.sum()) + prompt * start + prompt * (prompt + 1) // 2
        return dict(bytes=layers * (mats * 2 + (cached + n) * 2 * KVDIM * 2) + vocab * HIDDEN * 2
                    + 2 * n * HIDDEN * 2 + nl * vocab * 2,
                    flops=layers * (2 * n * mats + 4 * pairs * QDIM) + 2 * nl * vocab * HIDDEN)

    @classmethod
    def exact(cls, case, seed):
        rows, cfg = _Row(case, seed), _model(case)
        embed, final_norm, layers = weights.engine_layers(_model_weights(case, seed), cfg)
        inv, pos = _inv_freq(), _ints(rows.positions)
        d, n = rows.decode, rows.n
        tables = _ints(rows.seq_tables).long()
        own = _ints(rows.tables).long()
        at = own.gather(1, (pos.long() // PAGE)[:, None])[:, 0] * PAGE + pos % PAGE
        ends = [int(x) for x in rows.lens]
        if rows.prompt:
            ends.append(rows.prompt + rows.start)
        seq_rows = []
        for b, m in enumerate(ends):
            i = torch.arange(m, device=DEV)
            seq_rows.append(tables[b][i // PAGE] * PAGE + i % PAGE)
        mask = (torch.arange(rows.prompt + rows.start, device=DEV)[None, :]
                > pos[d:, None]) if rows.prompt else None
        x = embed[torch.from_numpy(rows.tokens).long().to(DEV)].double()
        pools = dict(k_pool=[], v_pool=[])
        for l, w in enumerate(layers):
            h = _rmsnorm64(x, w["attn_norm"])
            q = _rope64((h @ w["wq"].double().t()).view(n, HEADS, HEAD), pos, inv)
            k = _rope64((h @ w["wk"].double().t()).view(n, KV_HEADS, HEAD), pos, inv)
            v = h @ w["wv"].double().t()
            kp, vp = (t.view(-1, KVDIM).double() for t in _fill(case, rows, l, seed))
            kp[at], vp[at] = k.reshape(n, KVDIM), v
            out = torch.empty((n, HEADS, HEAD), dtype=torch.float64, device=DEV)
            for b, r in enumerate(seq_rows):
                to, m = (slice(b, b + 1), None) if b < d else (slice(d, n), mask)
                out[to] = _attend64(q[to], kp[r].view(-1, KV_HEADS, HEAD),
                                    vp[r].view(-1, KV_HEADS, HEAD), m)
            x = x + out.view(n, QDIM) @ w["wo"].double().t()
            h = _rmsnorm64(x, w["mlp_norm"])
            act = _swiglu64(h @ w["w_gate"].double().t(), h @ w["w_up"].double().t())
            x = x + act @ w["w_down"].double().t()
            if case["kind"] == "block":
                pools["k_pool"].append(kp)
                pools["v_pool"].append(vp)
        pick = x if rows.logit_rows is None else x[torch.from_numpy(rows.logit_rows).long().to(DEV)]
        logits = _rmsnorm64(pick, final_norm) @ embed.double().t()
        out = dict(logits=logits, residual=x)
        if case["kind"] == "block":
            out.update(pools)
        return out

    @staticmethod
    def tolerance(case):
        return {"rel": 6e-3, "max": 1e-1} if case["kind"] == "block" else {"rel": 1.5e-2, "max": 2e-1}


_KINDS = dict(add_rmsnorm=_AddRmsnorm, swiglu=_Swiglu, nongemm_pass=_NongemmPass,
              attention=_Attention, mlp=_Mlp, block=_Forward, step=_Forward)
