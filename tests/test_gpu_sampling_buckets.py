"""Nucleus sampling's first-level buckets and the split below which elements
only add to a sum (sample.hip).

Two bars: equal tokens wherever the oracle's margin exceeds 1e-5 (as in
test_gpu_sampling.py), and at every row, whatever its margin, a token whose
running share holds tau (in_reach).
"""
from fractions import Fraction

import numpy as np
import pytest

import oracle as O
from mesh_amd.provider import sample_device
from tests.test_gpu_sampling import MARGIN, _check, _ctx

SPLIT = np.float32(2.0 ** -14)


def exponents(x, temperature):
    """(y - max) log2 e in f32, y the logits over the temperature."""
    t = np.float32(temperature)
    y = x * (np.float32(1) / t) if t != 1 else x
    return (y - y.max()) * np.float32(1.44269504088896341)


def nucleus(e, top_p, seeds):
    """[(token, e of the token)] per seed and e of the last kept element:
    elements by (e descending, column ascending), the last kept one the first
    whose running weight reaches top_p of the whole, the token the first to
    reach tau of the kept weight."""
    w = np.floor(e.astype(np.float64) * 2.0 ** 36 + 0.5).astype(np.int64)
    order = np.argsort(-e, kind="stable")
    cum = np.cumsum(w[order])

    def first(target):  # a Fraction
        return min(int(np.searchsorted(cum, -(-target.numerator // target.denominator))), e.size - 1)

    last = first(Fraction(float(np.float32(top_p))) * int(cum[-1]))
    hits = [first(Fraction(O.sample_threshold(int(s))) * int(cum[last])) for s in seeds]
    return [(int(order[h]), e[order[h]]) for h in hits], e[order[last]]


def in_reach(x, temperature, top_p, seed, token):
    """The token's running share, in float64, holds tau.

    e is off by (1 + |y - max|) 2^-23 of its value, its weight by 2^-37: sums of
    up to 128256 of them, almost all of their mass at |y - max| < 20, are off by
    less than 5e-6 of the whole (2.4e-6 + 128256 x 2^-37 + f64 rounding), which
    moves the kept mass and both ends; elements closer to the token's than twice
    the error of e may lie on either side of it."""
    d = exponents(x, temperature).astype(np.float64)
    p = np.exp2(d)
    p /= p.sum()
    if p[token] == 0:
        return False
    cum = np.cumsum(np.sort(p)[::-1])
    eps, last = 5e-6, len(p) - 1
    kept = [cum[min(int(np.searchsorted(cum, float(np.float32(top_p)) + z)), last)] for z in (-eps, eps)]
    near = 2 * 2.0 ** -23 * (1 - d[token])
    above, through = p[p > p[token] * (1 + near)].sum(), p[p >= p[token] * (1 - near)].sum()
    tau = O.sample_threshold(int(seed))
    return (above - eps) / kept[1] <= tau <= (through + eps) / kept[0]


def rows_of(kind, rng, cols):
    x = rng.standard_normal(cols).astype(np.float32)
    if kind == "peaked":                       # a language model's row: few tokens hold the mass
        x = x * 2
        n = min(20, cols)
        x[rng.permutation(cols)[:n]] += np.linspace(8, 14, n, dtype=np.float32)
    elif kind == "flat":                       # every element above the split
        x = x * np.float32(0.2)
    elif kind == "one_token":                  # the crossing below the split: one token holds half of the mass
        x = x * np.float32(0.1)
        x[rng.integers(cols)] = np.log(np.float32(cols))
    elif kind == "two_heights":                # a plateau right at the split, one right below it
        x = np.where(rng.random(cols) < 0.5, -np.float32(14 * np.log(2.0)), -np.float32(14.02 * np.log(2.0)))
        x[rng.permutation(cols)[:3]] = 0.0
        x = x.astype(np.float32)
    elif kind == "masked":
        x[rng.permutation(cols)[: cols - max(2, cols // 50)]] = -np.inf
    elif kind == "steps":                      # powers of two apart: every element on a bucket's edge
        x = (-np.float32(np.log(2.0)) * rng.integers(0, 30, cols)).astype(np.float32)
    elif kind == "ties":
        x = np.round(x * 3) / np.float32(3)
    return x


def tail_row(rng, cols):
    """One element at e = 1 and about 3000 a little below the split, each 3 to
    5e-5 of the mass: wide enough for a draw among them to be told apart."""
    x = np.full(cols, -np.inf, np.float32) if rng.random() < 0.5 else rng.uniform(-40, -30, cols).astype(np.float32)
    n = min(cols - 1, 3000)
    at = rng.permutation(cols)[:n + 1]
    x[at[:n]] = np.log(rng.uniform(0.5, 0.95, n) * float(SPLIT)).astype(np.float32)
    x[at[n]] = 0
    return x


def tail_draws(cols, rows):
    """Rows whose last kept element and whose draw both lie below the split,
    and whose draw the oracle can tell apart."""
    rng = np.random.default_rng(cols)
    x, temps, tops, seeds = [], [], [], []
    while len(x) < rows:
        t, p = np.float32(rng.choice([1.0, 0.7, 1.3])), np.float32(rng.uniform(0.95, 0.99))
        row = (tail_row(rng, cols) * t).astype(np.float32)
        some = rng.integers(0, 2 ** 63, 200, dtype=np.uint64)
        drawn, last = nucleus(np.exp2(exponents(row, t)), p, some)
        low = [s for s, (_, e) in zip(some, drawn) if e < SPLIT and last < SPLIT]
        for seed in low[:3]:
            if O.sample_token_device(row, float(t), float(p), int(seed))[1] > MARGIN:
                x.append(row)
                temps.append(t)
                tops.append(p)
                seeds.append(seed)
                break
    return np.stack(x), np.array(temps, np.float32), np.array(tops, np.float32), np.array(seeds, np.uint64)


def test_whole_number_rule_is_the_oracles():
    """The restatement, with numpy's exp2, against the oracle at the rows it can tell apart."""
    x, temps, tops, seeds = tail_draws(4096, 12)
    rng = np.random.default_rng(1)
    rows = list(zip(x, temps, tops, seeds))
    for k in ("peaked", "one_token", "masked", "ties"):
        rows += [(rows_of(k, rng, 1023), np.float32(0.7), np.float32(0.9), s) for s in rng.integers(0, 2 ** 63, 8)]
    compared = 0
    for row, t, p, s in rows:
        want, margin = O.sample_token_device(row, float(t), float(p), int(s))
        if margin > MARGIN:
            assert nucleus(np.exp2(exponents(row, t)), p, [s])[0][0][0] == want
            compared += 1
        # the oracle's own token is in reach, one that sorts far from it is not
        assert in_reach(row, t, p, s, want)
        order = np.argsort(-row, kind="stable")
        share = np.cumsum(np.exp2(exponents(row, t).astype(np.float64))[order])
        far = order[int(np.searchsorted(share, (share[np.where(order == want)[0][0]] + 0.3 * share[-1]) % share[-1]))]
        assert far == want or not in_reach(row, t, p, s, int(far))
    assert compared >= 36


@pytest.mark.gpu
@pytest.mark.parametrize("cols", [128256, 32000, 9001, 3001])
def test_draws_below_the_split(cols):
    """The top_p crossing and the drawn token both below the split: the second
    pass's buckets decide the token."""
    ctx = _ctx(cols)
    x, temps, tops, seeds = tail_draws(cols, 24)
    got = sample_device(ctx, x, temps, tops, seeds)
    assert _check(x, temps, tops, seeds, got) == len(x)
    ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("cols", [128256, 32000, 9001, 4096, 1023, 40])
@pytest.mark.parametrize("kind", ["peaked", "flat", "one_token", "two_heights", "masked", "steps", "ties"])
def test_rows_of_every_shape_match_oracle(cols, kind):
    ctx = _ctx(cols)
    rng = np.random.default_rng(cols + len(kind))
    rows = 24
    x = np.stack([rows_of(kind, rng, cols) for _ in range(rows)])
    temps = rng.choice([1.0, 0.7, 1.3, 0.25], rows).astype(np.float32)
    tops = rng.choice([0.999, 0.95, 0.9, 0.5, 0.01], rows).astype(np.float32)
    seeds = rng.integers(0, 2 ** 63, rows, dtype=np.uint64)
    got = sample_device(ctx, x, temps, tops, seeds)
    compared = _check(x, temps, tops, seeds, got)
    # (flat rows of many columns: every probability is near 1e-5, every draw within the margin of a boundary)
    assert compared >= rows // 3 or (kind not in ("peaked", "masked") and cols > 1000), compared
    for r in range(rows):
        assert in_reach(x[r], temps[r], tops[r], seeds[r], got[r]), r
    assert sample_device(ctx, x, temps, tops, seeds) == got
    ctx.close()
