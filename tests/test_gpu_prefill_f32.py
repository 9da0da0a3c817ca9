"""Prefill chunks over f32 pools (paged_prefill_attention_f32_kernel) against a
float64 restatement.

Tolerance: Q, P, K and V enter the products as bf16 hi + lo, each off by at
most 2^-17 of its value, and the lo x lo products (2^-17 again) are left out; a
score of D products of N(0, 1) values then moves by about 2^-16 / sqrt(d) times
sqrt(D), i.e. ~2e-5, and the weighted sum as much: 1e-4 of a row's largest
value leaves a factor of three."""
import ctypes as C

import numpy as np
import pytest

from mesh_amd import DeviceContext, KVCacheSnapshot, ModelGeometry, _lib
from tests.gpu_util import stage_mixed
from tests.test_gpu_attention_plain import reference, run_attention

pytestmark = pytest.mark.gpu

RTOL = 1e-4


def worst(out, want, heads, D):
    d = np.abs(out - want).reshape(len(out), heads, D).max(-1)
    return (d / np.abs(want).reshape(len(out), heads, D).max(-1)).max()


@pytest.mark.parametrize("key_halves,tiles_per_split", [("1", "2"), ("2", "2"), ("2", "3"), ("2", None), ("1", None)])
@pytest.mark.parametrize("heads,kv_heads,D", [(8, 8, 64), (8, 4, 128), (32, 8, 128), (16, 2, 64), (16, 1, 128)])
def test_chunks_of_every_group_and_split(monkeypatch, heads, kv_heads, D, key_halves, tiles_per_split):
    """Chunks of 128 / G rows (the shortest that leaves the decode tiles, with
    enough visible keys) and one row less, ragged blocks, page-unaligned and
    trimmed windows, decode rows beside them; whole blocks and key splits of 2
    and 3 tiles."""
    if tiles_per_split:
        monkeypatch.setenv("ZR_ATTN_PREFILL_TILES_PER_SPLIT", tiles_per_split)
    monkeypatch.setenv("ZR_ATTN_PREFILL_KEY_HALVES", key_halves)
    rows = 128 * kv_heads // heads
    cases = [(0, rows, 0), (1603, rows, 0), (903, 2 * rows + 5, 0), (1700, rows - 1, 0), (77, 1, 0),
             (1601, rows + 1, 9)]
    out, seqs = run_attention(heads, kv_heads, D, "f32", cases, np.random.default_rng(D + heads))
    assert worst(out, reference(seqs, heads, kv_heads, D), heads, D) <= RTOL


@pytest.mark.parametrize("key_halves", ["1", "2"])
@pytest.mark.parametrize("heads,kv_heads,D", [(32, 4, 64), (32, 8, 128)])
def test_rows_a_query_does_not_see_never_reach_it(monkeypatch, heads, kv_heads, D, key_halves):
    """Values that are not finite in the chunk's later rows, in rows trimmed off
    the window and in what an earlier owner left in its pages reach only the
    queries that see them."""
    monkeypatch.setenv("ZR_ATTN_PREFILL_KEY_HALVES", key_halves)
    cases = [(840, 70, 7), (20, 1, 0)]

    def stale(ctx):
        owner = ctx.new_backend()
        n = 16 * ctx.lib.zr_kv_pool_pages(ctx.h)
        x = np.full((1, n, kv_heads * D), np.inf, np.float32)
        owner.import_kv_cache(KVCacheSnapshot(n, n, x, x))
        owner.release_pages()

    def edit(Ks, Vs):
        Vs[0][:7] = np.nan
        Vs[0][7 + 840 + 31, 5] = np.inf
        Vs[0][7 + 840 + 52, D + 3] = -np.inf

    out, seqs = run_attention(heads, kv_heads, D, "f32", cases, np.random.default_rng(4), edit, stale)
    with np.errstate(invalid="ignore"):
        want = reference(seqs, heads, kv_heads, D)
    fine = np.isfinite(want)[:70]
    assert fine[:31].all() and not fine[31:].all()
    np.testing.assert_array_equal(np.isfinite(out)[:70], fine)
    np.testing.assert_allclose(out[:70][fine], want[:70][fine], rtol=0, atol=RTOL * np.abs(want[:70][fine]).max())


@pytest.mark.parametrize("heads,kv_heads,D", [(32, 4, 64), (16, 8, 128)])
def test_read_probe_of_prompt_chunks_alone(heads, kv_heads, D):
    """zr_kv_read_probe takes a microbatch of chunks alone from an f32 pool,
    whether they have the work for prefill blocks (600 rows on 1500) or stay on
    decode tiles (20 rows), and leaves the pages as they were; from a bf16 pool
    such a microbatch has no decode items."""
    for kv_dtype, chunks, status in (("f32", [600, 601], _lib.ZR_OK), ("f32", [20], _lib.ZR_OK),
                                     ("bf16", [600, 601], _lib.ZR_E_INVALID)):
        geo = ModelGeometry(hidden=heads * D, num_heads=heads, num_kv_heads=kv_heads, num_layers=1, vocab=32, ffn=32)
        ctx = DeviceContext(geo, kv_dtype=kv_dtype, max_tokens=1201, max_seqs=2, max_pages_per_seq=200)
        ctx.create_kv_pool(300)
        x = np.random.default_rng(D).standard_normal((1, 1500, kv_heads * D), dtype=np.float32)
        backends = [ctx.new_backend() for _ in chunks]
        for b in backends:
            b.import_kv_cache(KVCacheSnapshot(1500, 1500, x, -x))
        st = stage_mixed(ctx, backends, chunks)
        before = [b.export_kv_cache() for b in backends]
        ms = C.c_double()
        assert ctx.lib.zr_kv_read_probe(ctx.h, st, 0, 5, C.byref(ms)) == status
        if status == _lib.ZR_OK:
            assert 0.0 < ms.value < 100.0
        ctx.lib.zr_staged_destroy(st)
        for b, snap in zip(backends, before):
            after = b.export_kv_cache()
            np.testing.assert_array_equal(after.keys, snap.keys)
            np.testing.assert_array_equal(after.values, snap.values)
        ctx.close()
