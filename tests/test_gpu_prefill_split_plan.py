"""The size of prefill attention's key splits (zr::prefill_tiles_per_split):
its workgroups against the resident slots on the CPU, and chunks that take one
and two passes against a float64 restatement."""
import ctypes as C

import numpy as np
import pytest

from mesh_amd import _lib
from tests.test_gpu_attention_plain import reference, run_attention
from tests.test_gpu_prefill_f32 import RTOL, worst

SLOTS = 256          # 8-wave workgroups, one per CU
PASS, MERGE = 8, 10  # prices in tiles


def block_tiles(chunks, rows_per_block):
    """32-key tiles of each block; chunks of (rows, rows before them)."""
    return [((before + min(r0 + rows_per_block, rows) + 15) // 16 + 1) // 2
            for rows, before in chunks for r0 in range(0, rows, rows_per_block)]


def split_size(tiles, kv_heads, slots=SLOTS):
    fn = C.CDLL(_lib.LIB_PATH)._ZN2zr23prefill_tiles_per_splitEPKiiii
    fn.restype, fn.argtypes = C.c_int, [C.c_void_p, C.c_int, C.c_int, C.c_int]
    return fn((C.c_int * max(len(tiles), 1))(*tiles), len(tiles), kv_heads, slots)


def workgroups(tiles, kv_heads, size):
    return sum(-(-t // size) for t in tiles) * kv_heads


def price(tiles, kv_heads, size, slots=SLOTS):
    longest = max(tiles)
    if size >= longest:
        return longest + PASS
    piece = max(-(-t // -(-t // size)) for t in tiles)  # a block's splits are even
    return -(-workgroups(tiles, kv_heads, size) // slots) * (piece + PASS) + MERGE


# rows, rows before them, kv heads, rows per block, passes (0: blocks whole)
PLANS = [(32, 2000, 8, 32, 1), (40, 500, 8, 32, 1), (300, 500, 8, 32, 1), (400, 1200, 8, 32, 1), (600, 500, 8, 32, 1),
         (600, 0, 8, 32, 0), (700, 500, 8, 32, 0), (900, 0, 8, 32, 0), (1000, 0, 4, 16, 0), (512, 0, 4, 16, 0),
         (600, 1200, 8, 32, 2), (544, 6000, 8, 32, 2)]


@pytest.mark.parametrize("rows,before,kv_heads,rows_per_block,passes", PLANS)
def test_splits_fill_whole_passes(rows, before, kv_heads, rows_per_block, passes):
    tiles = block_tiles([(rows, before)], rows_per_block)
    size = split_size(tiles, kv_heads)
    if passes == 0:
        assert size >= max(tiles)
    else:
        assert size < max(tiles)
        assert -(-workgroups(tiles, kv_heads, size) // SLOTS) == passes


def test_no_size_within_two_passes_is_cheaper():
    rng = np.random.default_rng(0)
    for _ in range(400):
        kv_heads, per = [(8, 32), (4, 32), (4, 16), (8, 128), (1, 8)][rng.integers(5)]
        chunks = [(int(rng.integers(per, 1000)), int(rng.integers(0, 7000))) for _ in range(rng.integers(1, 4))]
        tiles = block_tiles(chunks, per)
        slots = int(rng.choice([256, 512]))
        size = split_size(tiles, kv_heads, slots)
        if len(tiles) * kv_heads >= slots:
            assert size >= max(tiles)
            continue
        assert size >= max(8, -(-max(tiles) // 16))
        least = max(8, -(-max(tiles) // 16))
        sizes = [s for s in range(least, max(tiles) + 1) if workgroups(tiles, kv_heads, s) <= 2 * slots]
        best = min([price(tiles, kv_heads, s, slots) for s in sizes] + [max(tiles) + PASS])
        assert price(tiles, kv_heads, size, slots) == best, (chunks, kv_heads, per, slots)


def test_no_blocks_and_one_tile():
    assert split_size([], 8) >= 1
    assert split_size([1], 1) >= 1
    assert split_size([1 << 20], 1) == 1 << 16  # 16 splits at most


@pytest.mark.gpu
@pytest.mark.parametrize("rows,before,passes", [(300, 500, 1), (1280, 1800, 2)])
def test_chunks_of_planned_splits(monkeypatch, rows, before, passes):
    """16 kv heads of 64, blocks of 128 rows, a decode row beside them."""
    monkeypatch.delenv("ZR_ATTN_PREFILL_TILES_PER_SPLIT", raising=False)
    tiles = block_tiles([(rows, before)], 128)
    assert -(-workgroups(tiles, 16, split_size(tiles, 16)) // SLOTS) == passes
    assert split_size(tiles, 16) < max(tiles)
    out, seqs = run_attention(16, 16, 64, "f32", [(before, rows, 0), (77, 1, 0)], np.random.default_rng(rows))
    assert worst(out, reference(seqs, 16, 16, 64), 16, 64) <= RTOL
