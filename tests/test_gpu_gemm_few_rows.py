"""Products of at most 8 rows: the weights straight to registers.

Every row count's edge (1, 2, 4, 8 rows and between; 9 take the tiles), k from a single
step (most waves have none) to several steps per wave and several workgroups
along K, columns that end inside a 16-column tile.
"""
import numpy as np
import pytest

import oracle as O
from mesh_amd import DeviceBuffer, DeviceContext, ModelGeometry, bf16_bits

pytestmark = pytest.mark.gpu


def context(split):
    geo = ModelGeometry(hidden=256, num_heads=4, num_kv_heads=4, num_layers=1, vocab=64, ffn=256)
    return DeviceContext(geo, kv_dtype="f32", max_tokens=16, max_seqs=4, max_pages_per_seq=4, split_activations=split)


def operand(a, split):
    """What the kernel multiplies: a as bf16 hi + lo, or bf16."""
    hi = O.round_bf16(a)
    return hi.astype(np.float64) + (O.round_bf16(a - hi).astype(np.float64) if split else 0.0)


def bound(a, w, k):
    # f32 sums of 2 k products in any order: (2 k + 16) 2^-24 of the sum of magnitudes
    return (2 * k + 16) * 2.0 ** -24 * (np.abs(a) @ np.abs(w)) + 1e-30


@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("m,k,n", [(1, 32, 16), (1, 2048, 2560), (2, 96, 100), (3, 2048, 2048), (5, 288, 33),
                                   (8, 5632, 2048), (8, 64, 4100), (9, 320, 100), (4, 14336, 4096)])
def test_store(split, m, k, n):
    ctx = context(split)
    rng = np.random.default_rng(m + k + n)
    a = rng.standard_normal((m, k), dtype=np.float32)
    w = O.round_bf16(rng.standard_normal((k, n), dtype=np.float32) * 0.02)
    wb = bf16_bits(w)
    d_a, d_c = DeviceBuffer.from_numpy(ctx, a), DeviceBuffer(ctx, m * n * 4)
    ctx.check(ctx.lib.zr_gemm(ctx.h, d_a.ptr, wb.ctypes.data, d_c.ptr, m, n, k))
    got = d_c.download(np.float32, (m, n))
    a64, w64 = operand(a, split), w.astype(np.float64)
    assert np.all(np.abs(got - a64 @ w64) <= bound(a64, w64, k))
    ctx.close()


@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("m,k,f", [(1, 32, 32), (1, 2048, 5632), (2, 96, 64), (3, 288, 128), (7, 352, 96), (8, 4096, 1024)])
def test_swiglu(split, m, k, f):
    ctx = context(split)
    rng = np.random.default_rng(m + k + f)
    a = rng.standard_normal((m, k), dtype=np.float32)
    wg, wu = (O.round_bf16(rng.standard_normal((k, f), dtype=np.float32) * 0.02) for _ in range(2))
    wgb, wub = bf16_bits(wg), bf16_bits(wu)
    d_a, d_h = DeviceBuffer.from_numpy(ctx, a), DeviceBuffer(ctx, m * f * 4)
    ctx.check(ctx.lib.zr_gemm_swiglu(ctx.h, d_a.ptr, wgb.ctypes.data, wub.ctypes.data, d_h.ptr, m, f, k))
    got = d_h.download(np.float32, (m, f))
    a64 = operand(a, split)
    g, u = a64 @ wg.astype(np.float64), a64 @ wu.astype(np.float64)
    ref = g / (1.0 + np.exp(-g)) * u
    # |silu'| <= 1.1, |silu(g)| <= |g|; a few roundings of silu and the product;
    # h is held as hi + lo (2^-16) or bf16 (2^-8)
    eg, eu = bound(a64, wg.astype(np.float64), k), bound(a64, wu.astype(np.float64), k)
    tol = 1.1 * eg * (np.abs(u) + eu) + np.abs(g) * eu + (2.0 ** -15 if split else 2.0 ** -8) * np.abs(ref) + 1e-30
    assert np.all(np.abs(got - ref) <= tol)
    ctx.close()


@pytest.mark.parametrize("m", [1, 7])
def test_other_rows_and_columns_do_not_matter(m):
    # infinities and NaN reach only their own row (of a) and column (of w)
    ctx = context(True)
    k, n = 256, 40
    rng = np.random.default_rng(m)
    a = rng.standard_normal((m, k), dtype=np.float32)
    w = O.round_bf16(rng.standard_normal((k, n), dtype=np.float32))
    w[5, 17], w[200, 39] = np.inf, np.nan
    if m > 1:
        a[m - 1, 7] = np.nan
    wb = bf16_bits(w)
    d_a, d_c = DeviceBuffer.from_numpy(ctx, a), DeviceBuffer(ctx, m * n * 4)
    ctx.check(ctx.lib.zr_gemm(ctx.h, d_a.ptr, wb.ctypes.data, d_c.ptr, m, n, k))
    bad = ~np.isfinite(d_c.download(np.float32, (m, n)))
    want = np.zeros((m, n), bool)
    want[:, [17, 39]] = True
    if m > 1:
        want[m - 1] = True
    assert np.array_equal(bad, want)
    ctx.close()
