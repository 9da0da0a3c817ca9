"""Nucleus sampling's first-level buckets and the split below which elements
only add to a sum (sample.hip), against the oracle's restatement (the bar of
test_gpu_sampling.py: equal tokens wherever the oracle's margin exceeds 1e-5)."""
import numpy as np
import pytest

from mesh_amd.provider import sample_device
from tests.test_gpu_sampling import _check, _ctx

pytestmark = pytest.mark.gpu


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
    assert sample_device(ctx, x, temps, tops, seeds) == got
    ctx.close()
