"""Attention over plain-layout pools (head_dim other than 64 / 128, or q heads
per kv head not dividing 16) against a float64 restatement: column tiles for a
head_dim that is a multiple of 4 (attention_plain.hip), one wave per row and q
head for the others (attention.hip's paged_attention_generic_kernel).

Tolerance: every product and sum is f32, as in the reference; a score of D
products and a weighted sum of L values carry a few rounding errors of 2^-24 of
their running magnitude.  1e-5 of a row's largest value is over ten times that
at D = 256 and 700 keys, and far below the 2^-16 of a bf16 hi + lo product."""
import ctypes as C
import math

import numpy as np
import pytest

from mesh_amd import DeviceBuffer, DeviceContext, KVCacheSnapshot, ModelGeometry, _lib
from tests.gpu_util import stage_mixed

RTOL = 1e-5


class PlainPlan(C.Structure):
    """zr::PlainAttnPlan (zr_internal.h)."""
    _fields_ = [("ct", C.c_int), ("waves", C.c_int)]


def plain_plan(heads, kv_heads, D, q_len):
    fn = C.CDLL(_lib.LIB_PATH)._ZN2zr20plain_attention_planEiiiPKii
    fn.restype = PlainPlan
    return fn(D, kv_heads, heads // kv_heads, (C.c_int * len(q_len))(*q_len), len(q_len))


def bf16(x):
    u = np.ascontiguousarray(x, np.float32).view(np.uint32).astype(np.uint64)
    return ((((u + 0x7FFF + ((u >> 16) & 1)) >> 16) << 16).astype(np.uint32)).view(np.float32)


def run_attention(heads, kv_heads, D, kv_dtype, cases, rng, edit=None, before=None):
    """(output, [(q, k, v, prefix)]) of one microbatch; cases are (window, chunk, rows trimmed before the window).
    `edit(Ks, Vs)` changes the rows first; `before(ctx)` runs on the fresh pool."""
    Q, KV = heads * D, kv_heads * D
    geo = ModelGeometry(hidden=Q, num_heads=heads, num_kv_heads=kv_heads, num_layers=1, vocab=32, ffn=32)
    T = sum(c for _, c, _ in cases)
    ctx = DeviceContext(geo, kv_dtype=kv_dtype, max_tokens=T, max_seqs=len(cases), max_pages_per_seq=200)
    ctx.create_kv_pool(sum((t + p + c + 15) // 16 + 1 for p, c, t in cases))
    if before:
        before(ctx)
    Ks = [rng.standard_normal((t + p + c, KV), dtype=np.float32) for p, c, t in cases]
    Vs = [rng.standard_normal((t + p + c, KV), dtype=np.float32) for p, c, t in cases]
    if edit:
        edit(Ks, Vs)
    backends = []
    for (p, c, t), k, v in zip(cases, Ks, Vs):
        b = ctx.new_backend()
        if t + p:
            b.import_kv_cache(KVCacheSnapshot(t + p, t + p, k[None, :t + p], v[None, :t + p]))
        if t:
            b.retain_suffix(p)
        backends.append(b)
    Qm = rng.standard_normal((T, Q), dtype=np.float32)
    new = [np.concatenate([x[t + p:] for x, (p, _, t) in zip(xs, cases)]) for xs in (Ks, Vs)]
    st = stage_mixed(ctx, backends, [c for _, c, _ in cases])
    d_qkv = DeviceBuffer.from_numpy(ctx, np.concatenate([Qm] + new, 1))
    d_q, d_o = DeviceBuffer(ctx, Qm.nbytes), DeviceBuffer(ctx, Qm.nbytes)
    ctx.check(ctx.lib.zr_rope_kv_write(ctx.h, st, 0, d_qkv.ptr, d_q.ptr, 0))
    ctx.check(ctx.lib.zr_attention(ctx.h, st, 0, d_q.ptr, d_o.ptr))
    out = d_o.download(np.float32, Qm.shape)
    ctx.lib.zr_staged_destroy(st)
    ctx.close()
    seqs, row = [], 0
    for (p, c, t), k, v in zip(cases, Ks, Vs):
        k, v = k[t:], v[t:]
        if kv_dtype == "bf16":
            k, v = bf16(k), bf16(v)
        seqs.append((Qm[row:row + c], k, v, p))
        row += c
    return out, seqs


def reference(seqs, heads, kv_heads, D):
    rows = []
    for q, k, v, p in seqs:
        for r in range(q.shape[0]):
            n = p + r + 1
            ks = k[:n].astype(np.float64).reshape(n, kv_heads, D)
            vs = v[:n].astype(np.float64).reshape(n, kv_heads, D)
            qs = q[r].astype(np.float64).reshape(kv_heads, heads // kv_heads, D)
            s = np.einsum("hgd,nhd->hgn", qs, ks) / math.sqrt(D)
            w = np.exp(s - s.max(-1, keepdims=True))
            w /= w.sum(-1, keepdims=True)
            rows.append(np.einsum("hgn,nhd->hgd", w, vs).reshape(-1))
    return np.stack(rows)


@pytest.mark.gpu
@pytest.mark.parametrize("kv_dtype", ["f32", "bf16"])
@pytest.mark.parametrize("heads,kv_heads,D", [
    (8, 8, 4), (8, 4, 16), (8, 2, 20), (8, 8, 36), (8, 1, 48), (8, 2, 60), (8, 8, 80), (8, 4, 96), (8, 2, 100),
    (8, 8, 112), (28, 4, 128), (8, 4, 132), (8, 8, 160), (8, 4, 192), (8, 2, 256), (6, 2, 64), (64, 2, 64)])
def test_every_multiple_of_four_head_dim_and_group(kv_dtype, heads, kv_heads, D):
    """Decode rows and chunks, windows trimmed to start mid-page, one-key
    windows; head dims on both sides of every block of 16 and group of 64; 1
    to 32 q heads per kv head."""
    cases = [(0, 1, 0), (0, 37, 0), (300, 1, 0), (57, 20, 9), (16, 1, 0), (130, 1, 5)]
    out, seqs = run_attention(heads, kv_heads, D, kv_dtype, cases, np.random.default_rng(D * heads + kv_heads))
    want = reference(seqs, heads, kv_heads, D)
    err = np.abs(out - want).reshape(len(out), heads, D).max(-1) / np.abs(want).reshape(len(out), heads, D).max(-1)
    assert err.max() <= RTOL, np.unravel_index(err.argmax(), err.shape)


@pytest.mark.gpu
@pytest.mark.parametrize("kv_dtype", ["f32", "bf16"])
@pytest.mark.parametrize("heads,kv_heads,D", [(16, 16, 2), (16, 4, 6), (48, 16, 18), (16, 2, 62), (16, 16, 66),
                                              (16, 2, 98), (16, 8, 126), (16, 16, 130), (16, 4, 190), (16, 2, 254)])
def test_even_head_dims_that_are_no_multiple_of_four(kv_dtype, heads, kv_heads, D):
    """The scalar kernel: a wave walks 64 keys at a time and holds up to 4 dims
    a lane, so windows end inside the first 64 keys, on the 64th and past it,
    and head dims on both sides of 64, 128 and 192."""
    cases = [(0, 1, 0), (0, 37, 0), (300, 1, 0), (57, 20, 9), (63, 2, 0), (130, 1, 5)]
    out, seqs = run_attention(heads, kv_heads, D, kv_dtype, cases, np.random.default_rng(D * heads + kv_heads))
    want = reference(seqs, heads, kv_heads, D)
    err = np.abs(out - want).reshape(len(out), heads, D).max(-1) / np.abs(want).reshape(len(out), heads, D).max(-1)
    assert err.max() <= RTOL, np.unravel_index(err.argmax(), err.shape)


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kv_heads,D,rows", [(32, 32, 80, 200), (32, 8, 96, 90), (16, 4, 256, 60)])
def test_wide_and_narrow_column_tiles(heads, kv_heads, D, rows):
    """Chunks beside decode rows: 32-column tiles, 16-column ones where wider
    ones would leave CUs idle, and the only form above 128 dims."""
    assert plain_plan(heads, kv_heads, D, [rows, 1]).ct == (2 if D == 80 else 1)
    out, seqs = run_attention(heads, kv_heads, D, "bf16", [(411, rows, 3), (690, 1, 0)], np.random.default_rng(rows))
    want = reference(seqs, heads, kv_heads, D)
    err = np.abs(out - want).reshape(len(out), heads, D).max(-1) / np.abs(want).reshape(len(out), heads, D).max(-1)
    assert err.max() <= RTOL


@pytest.mark.gpu
@pytest.mark.parametrize("kv_dtype", ["f32", "bf16"])
def test_rows_a_query_does_not_see_never_reach_it(kv_dtype):
    """Infinite and NaN values in rows outside a query's window: later rows of
    its chunk, rows trimmed off its first page, and what an earlier owner left
    in its pages.  Queries that see such a row get inf / NaN, all others stay
    finite and right."""
    heads, kv_heads, D = 8, 4, 80
    cases = [(40, 30, 7), (33, 1, 0), (20, 1, 6)]

    def stale(ctx):
        owner = ctx.new_backend()
        n = 16 * ctx.lib.zr_kv_pool_pages(ctx.h)
        n = min(n, 64 * 16)
        x = np.full((1, n, kv_heads * D), np.nan, np.float32)
        owner.import_kv_cache(KVCacheSnapshot(n, n, x, x))
        owner.release_pages()

    def edit(Ks, Vs):
        Vs[0][:7] = np.nan        # trimmed away
        Vs[0][7 + 40 + 11, 5] = np.inf  # the chunk's row 11
        Ks[2][:6] = np.inf

    out, seqs = run_attention(heads, kv_heads, D, kv_dtype, cases, np.random.default_rng(3), edit, stale)
    with np.errstate(invalid="ignore"):
        want = reference(seqs, heads, kv_heads, D)
    assert np.isfinite(want).sum() < want.size and np.isfinite(want[:11]).all() and np.isfinite(want[30:]).all()
    np.testing.assert_array_equal(np.isfinite(out), np.isfinite(want))
    fine = np.isfinite(want)
    np.testing.assert_allclose(out[fine], want[fine], rtol=0, atol=RTOL * np.abs(want[fine]).max())


# 32-column tiles: every count of 16-dim blocks they have, its first and its
# last head dim; (heads, kv heads, D, chunk rows, waves)
WIDE = [(32, 32, 4, 200, 8), (32, 32, 16, 200, 8), (32, 32, 20, 200, 8), (32, 32, 32, 200, 8), (32, 32, 36, 200, 8),
        (32, 32, 48, 200, 8), (32, 32, 52, 200, 8), (48, 16, 64, 200, 8), (32, 32, 68, 200, 8), (32, 32, 80, 212, 8),
        (32, 32, 84, 200, 8), (32, 32, 96, 200, 8), (32, 32, 100, 200, 8), (32, 32, 112, 220, 8),
        (32, 32, 116, 200, 4), (40, 8, 128, 220, 4), (64, 16, 40, 257, 4), (48, 16, 96, 400, 4)]


@pytest.mark.parametrize("heads,kv_heads,D,rows,waves", WIDE)
def test_wide_cases_take_the_tiles_they_name(heads, kv_heads, D, rows, waves):
    p = plain_plan(heads, kv_heads, D, [rows, 1])
    assert (p.ct, p.waves) == (2, waves)


@pytest.mark.gpu
@pytest.mark.parametrize("kv_dtype", ["f32", "bf16"])
@pytest.mark.parametrize("heads,kv_heads,D,rows,waves", WIDE)
def test_tiles_of_32_columns(kv_dtype, heads, kv_heads, D, rows, waves):
    """A chunk on a window trimmed to start mid-page, its last tile narrower
    than 16 columns or ending inside its second half, beside a decode row."""
    out, seqs = run_attention(heads, kv_heads, D, kv_dtype, [(150, rows, 3), (690, 1, 0)], np.random.default_rng(D))
    want = reference(seqs, heads, kv_heads, D)
    err = np.abs(out - want).reshape(len(out), heads, D).max(-1) / np.abs(want).reshape(len(out), heads, D).max(-1)
    assert err.max() <= RTOL, np.unravel_index(err.argmax(), err.shape)


@pytest.mark.gpu
@pytest.mark.parametrize("kv_dtype", ["f32", "bf16"])
@pytest.mark.parametrize("heads,kv_heads,D", [(32, 32, 20), (32, 32, 80), (48, 16, 96), (32, 32, 112), (40, 8, 128)])
def test_unseen_rows_in_tiles_of_32_columns(kv_dtype, heads, kv_heads, D):
    """As test_rows_a_query_does_not_see_never_reach_it, with both column
    tiles of a workgroup on the page."""
    rows = 240

    def edit(Ks, Vs):
        Vs[0][:7] = np.nan
        Vs[0][7 + 40 + 11, 5] = np.inf   # the chunk's row 11: columns of the first tiles see it or not
        Vs[0][7 + 40 + 150, 1] = -np.inf
        Ks[1][:6] = np.inf

    out, seqs = run_attention(heads, kv_heads, D, kv_dtype, [(40, rows, 7), (20, 1, 6)], np.random.default_rng(D), edit)
    with np.errstate(invalid="ignore"):
        want = reference(seqs, heads, kv_heads, D)
    assert plain_plan(heads, kv_heads, D, [rows, 1]).ct == 2
    assert np.isfinite(want[:11]).all() and not np.isfinite(want[11:rows]).all()
    np.testing.assert_array_equal(np.isfinite(out), np.isfinite(want))
    fine = np.isfinite(want)
    np.testing.assert_allclose(out[fine], want[fine], rtol=0, atol=RTOL * np.abs(want[fine]).max())
