"""Attention of a prompt's rows in tiles (csrc/attention_prompt.hip) against float64, through a
one-layer engine whose projections are exact: token vectors of equal magnitudes (the norm turns
them into signs), projections that are short sums of binary fractions, a RoPE that turns only the
pair (0, 32), which the queries leave out, an identity output projection and an MLP of zeros. The
residual is then x + attention, the keys and values are read back from the pools, and the queries
are known.

A row's result is rounded to fp16 twice (2^-11 each: the attention, then the residual sum) on top
of fp32 sums; 128 fp32 roundings (2^-17) of sum p |v| are allowed for these."""
import importlib

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
X = 2.0 ** -14  # magnitude of a token vector's elements


class Rows:
    """n rows of one sequence at positions start .. start + n - 1, each with a token of its own
    whose signs the caller may set, over cached keys and values that it gives."""

    def __init__(self, n_kv, n, start=0, seed=0):
        self.rng = np.random.default_rng(seed)
        self.n_kv, self.n, self.start, self.hidden = n_kv, n, start, 256 * n_kv
        self.signs = self.rng.choice([-1.0, 1.0], (n, self.hidden))
        self.signs[:, 0] = 1.0
        kvd = 64 * n_kv
        # one row per head: [dims, columns of the token vector]
        self.wq, self.wk, self.wv = (np.zeros((k, 64, self.hidden)) for k in (4 * n_kv, n_kv, n_kv))
        self.cached = [np.zeros((start, kvd), np.float16) for _ in range(2)]

    def run(self, llmk, capture=False):
        """(residual - x, keys, values), in float64."""
        h, n, n_kv = self.hidden, self.n, self.n_kv
        end = self.start + n
        pages = (end + 15) // 16
        cfg = llmk.ModelConfig(n_layers=1, hidden=h, n_heads=4 * n_kv, n_kv_heads=n_kv, inter=128,
                               vocab=n, eps=1e-15, rope_theta=1e300)
        half = lambda a: torch.from_numpy(np.ascontiguousarray(a).astype(np.float16)).cuda()
        x = self.signs * X
        e = llmk.Engine(cfg, n, pages, pages)
        e.set_weights(half(x), half(np.ones(h)), [dict(
            attn_norm=half(np.ones(h)), wq=half(self.wq.reshape(-1, h)),
            wk=half(self.wk.reshape(-1, h)), wv=half(self.wv.reshape(-1, h)), wo=half(np.eye(h)),
            mlp_norm=half(np.ones(h)), w_gate=half(np.zeros((128, h))),
            w_up=half(np.zeros((128, h))), w_down=half(np.zeros((h, 128))))])
        table = self.rng.permutation(pages).astype(np.int32)
        at = table[np.arange(end) // 16] * 16 + np.arange(end) % 16
        for which, rows in zip((llmk.BUF_K_POOL, llmk.BUF_V_POOL), self.cached):
            pool = np.full((pages * 16, 64 * n_kv), np.nan, np.float16)
            pool[at[:self.start]] = rows
            e.write_pool(which, 0, torch.from_numpy(pool.reshape(-1)))
        e.set_rows(np.arange(n, dtype=np.int32), np.arange(self.start, end, dtype=np.int32),
                   np.tile(table, (n, 1)), [n - 1])
        if capture:  # every row a decode row
            g, s = torch.cuda.CUDAGraph(), torch.cuda.Stream()
            torch.cuda.synchronize()
            with torch.cuda.graph(g, stream=s):
                e.forward(n, 1, stream=s)
            g.replay()
        else:
            e.forward(n, 1)
        torch.cuda.synchronize()
        k, v = (e.pool(w, 0).double().cpu().numpy().reshape(-1, 64 * n_kv)[at]
                for w in (llmk.BUF_K_POOL, llmk.BUF_V_POOL))
        return (e.residual(n).double().cpu().numpy().reshape(n, h) - x,
                k.reshape(end, n_kv, 64), v.reshape(end, n_kv, 64))

    def expected(self, k, v):
        """(attention, sum p |v|) of every row in float64, [n, 256 n_kv]."""
        out = np.empty((2, self.n, 4 * self.n_kv, 64))
        later = np.arange(self.start + self.n)[None, :] > self.start + np.arange(self.n)[:, None]
        for head in range(4 * self.n_kv):
            q = self.signs @ self.wq[head].T
            s = q @ np.nan_to_num(k[:, head // 4]).T / 8
            s[later] = -np.inf
            p = np.exp(s - s.max(-1, keepdims=True))
            p /= p.sum(-1, keepdims=True)
            vals = v[:, head // 4]
            out[0, :, head], out[1, :, head] = p @ vals, p @ np.abs(vals)
        return out.reshape(2, self.n, -1)

    def check(self, llmk, what=""):
        got, k, v = self.run(llmk)
        ref, spread = self.expected(k, v)
        assert_close(got, ref, spread, what)


def assert_close(got, ref, spread, what):
    bound = 2.0 ** -10 * np.abs(ref) + 2.0 ** -10 * X + 2.0 ** -17 * spread + 2.0 ** -24
    bad = ~(np.abs(got - ref) <= bound)
    assert not bad.any(), (what, int(bad.sum()), np.argwhere(bad)[:4], got[bad][:4], ref[bad][:4])


def random_rows(n_kv, n, start, seed):
    """Random queries, keys and values in binary fractions, the keys' part along the queries growing
    over the positions, so that the running maximum keeps rising (by 14 log2 units in all)."""
    r = Rows(n_kv, n, start, seed)
    r.wq[:, 1:5, 0] = 1.0
    r.wq[:, 33:63, 36:48] = r.rng.integers(-1, 2, (4 * n_kv, 30, 12)) / 4
    r.wk[:, 33:63, 20:36] = r.rng.integers(-1, 2, (n_kv, 30, 16)) / 4
    r.wv[:, :, 20:36] = r.rng.integers(-2, 3, (n_kv, 64, 16)) / 4
    # columns 1 to 15 count up from -1 to 1 over the positions
    level = (start + np.arange(n)) * 16 // (start + n)
    r.signs[:, 1:16] = np.where(level[:, None] >= np.arange(1, 16), 1.0, -1.0)
    r.wk[:, 1:5, 1:16] = 0.625
    if start:
        for rows, std in zip(r.cached, (0.75, 1.0)):
            rows[:] = r.rng.standard_normal(rows.shape) * std
        k = r.cached[0].reshape(start, n_kv, 64)
        k[:, :, 1:5] = 0.625 * 2 * (np.arange(start) * 16 // (start + n) - 7.5)[:, None, None]
    return r


# (kv heads, rows, first position), and what they launch: 8 waves over one step of one split, of
# several splits, and over 17 steps of one split (more than 512 blocks); 16 waves over four steps of
# one split, the last for half of them, and over splits of a step and a half.
EVERY_LAUNCH = [(1, 9, 0), (2, 70, 500), (3, 33, 700), (8, 2100, 0), (8, 1000, 0), (8, 1024, 1),
                (2, 33, 9000)]


@pytest.mark.parametrize("n_kv,n,start", EVERY_LAUNCH)
def test_every_launch(llmk, n_kv, n, start):
    random_rows(n_kv, n, start, seed=n + start).check(llmk, (n_kv, n, start))


@pytest.mark.parametrize("n_kv,n,start,odd", [(1, 40, 0, 20), (8, 1000, 0, 300), (8, 2100, 0, 2000),
                                              (2, 100, 500, 530)])
def test_rows_before_a_value_that_is_not_finite(llmk, n_kv, n, start, odd):
    """Position odd has an infinite value in one head: rows before it, in its tile and chunk as well,
    are as ever, rows from it on are not finite (the MLP spreads it over the row)."""
    r = random_rows(n_kv, n, start, seed=odd)
    r.signs[:, 50] = -1.0
    r.signs[odd - start, 50] = 1.0
    r.wv[0, 3, 0] = r.wv[0, 3, 50] = 40000.0
    got, k, v = r.run(llmk)
    assert np.isinf(v[odd, 0, 3]) and np.isfinite(v[start:odd]).all()
    ref, spread = r.expected(k, np.where(np.isfinite(v), v, 0.0))
    before = slice(0, odd - start)
    assert_close(got[before], ref[before], spread[before], odd)
    assert not np.isfinite(got[odd - start:]).any()


# (kv heads, rows, first position), and what they launch: 8 waves over one step; the same in three
# splits; 16 waves over several steps of one split, the last with wave sets that have no positions; 8
# waves over 17 steps.
LAUNCHES = [(1, 40, 0), (1, 300, 0), (8, 1000, 0), (8, 2100, 0)]


@pytest.mark.parametrize("n_kv,n,start", LAUNCHES)
@pytest.mark.parametrize("a,dims,qs,ks", [(128, 8, 4, 0.5), (3584, 8, 4, 2), (12288, 5, 16, 8),
                                          (12288, 20, 32, 16), (16384, 28, 32, 16),
                                          (24576, 10, 32, 16)])
def test_large_finite_scores(llmk, n_kv, n, start, a, dims, qs, ks):
    """Scores of 2^14.5 to 2^30.3 in units of log2: a weight's exponent is a small difference of
    large numbers, and a row's largest weight is 1 whichever way these round (by 4, 16 and 47 up
    and by 63 down in the last four). Every partial sum of q.k is exact, so the scores are too; they
    differ by multiples of 2 qs ks / 8."""
    r = Rows(n_kv, n, start, seed=a + n)
    r.wq[:, 1:1 + dims, 0] = r.wk[:, 1:1 + dims, 0] = a
    r.wq[:, 40:44, 0] = qs
    for d in range(4):
        r.wk[:, 40 + d, 16 + d] = ks
    r.wv[:, :, 20:36] = r.rng.integers(-4, 5, (n_kv, 64, 16)) / 8
    r.check(llmk, (a, dims))


@pytest.mark.parametrize("n_kv,n,start", LAUNCHES)
@pytest.mark.parametrize("key", [7.0, 9.75, 12.5])
def test_small_weights_keep_their_bits(llmk, n_kv, n, start, key):
    """Position 0 takes nearly all of every row's weight and its value is zero: the result is made
    of the others' weights, 2^-20, 2^-28 and 2^-36 of the largest, and their values near 2^14."""
    r = Rows(n_kv, n, start, seed=n + int(key))
    r.signs[:, 1] = 1.0
    r.signs[0, 1] = -1.0
    r.signs[0, 16:32:2], r.signs[0, 17:32:2] = 1.0, -1.0
    r.wq[:, 1:5, 0] = 2.0
    r.wk[:, 1:5, 1] = -key
    r.wq[:, 10:20, 0] = 0.5
    r.wk[:, 10:20, 16:26] = np.eye(10) / 2
    r.wv[:, :, 0] = r.wv[:, :, 1] = 2.0 ** 13
    pairs = r.rng.integers(0, 2, (n_kv, 64, 4)) * 2.0 ** 10
    r.wv[:, :, 16:24:2] = r.wv[:, :, 17:24:2] = pairs
    r.check(llmk, key)
