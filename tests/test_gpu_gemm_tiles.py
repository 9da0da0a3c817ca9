"""Products in the kernel form and tile that each case names, against float64.

Which form a product takes follows from its sizes alone (gemm_plan), so every
case states what it is there for and the plan is checked against that, without
a GPU too: a rule that moves a case to another form fails here instead of
leaving a form without a test.
"""
import ctypes as C

import numpy as np
import pytest

from mesh_amd import BackendMicrobatchExecutor, DeviceBuffer, KVCacheSnapshot, _lib
from tests import test_gpu_kernels as kernels
from tests.gpu_util import stage_mixed
from tests.test_gpu_model import make
from tests.testmodels import geometry, random_weights

STORE, SWIGLU = 0, 1


class GemmPlan(C.Structure):
    """zr::GemmPlan (zr_internal.h)."""
    _fields_ = [(n, C.c_int) for n in ("wm", "wn", "waves_m", "waves_n", "stages")] + [("few_rows", C.c_bool)] + \
               [(n, C.c_int) for n in ("KT", "NT", "row_blocks", "col_blocks", "splits", "kt_per_split")] + \
               [("direct", C.c_bool), ("ws_floats", C.c_size_t)]


def gemm_plan(m, n, k, epilogue, waits=True):
    """waits: of a call that waits for its microbatch, as zr_forward and zr_gemm_swiglu do."""
    fn = C.CDLL(_lib.LIB_PATH)._ZN2zr9gemm_planEiiiib
    fn.restype, fn.argtypes = GemmPlan, [C.c_int] * 4 + [C.c_bool]
    return fn(m, n, k, epilogue, waits)


def tile(p):
    return p.wm * p.waves_m * 32, p.wn * p.waves_n * 32


# (m, k, f, k-steps per wave of 4)
KSPLIT = [(9, 128, 64, 1), (15, 256, 96, 2), (31, 512, 1024, 4), (32, 2048, 5632, 16),  # one tile of 32 rows
          (33, 128, 64, 1), (45, 256, 96, 2), (63, 896, 512, 7)]                          # two


@pytest.mark.parametrize("m,k,f,steps", KSPLIT)
def test_ksplit_cases_take_the_launch_they_name(m, k, f, steps):
    p = gemm_plan(m, 2 * f, k, SWIGLU)
    assert (p.few_rows, p.waves_m, p.direct, p.splits, p.KT) == (False, 0, True, 1, 4 * steps)


@pytest.mark.gpu
@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("m,k,f,steps", KSPLIT)
def test_swiglu_with_k_over_four_waves(split, m, k, f, steps):
    """gemm_swiglu_ksplit_kernel: fewer steps per wave than its ring has
    stages, and rows that end inside a 32-row tile."""
    kernels.test_gemm_swiglu_matches_fp64(split, m, k, f)


# K steps that are no multiple of 4: (m, k, f, row tile, splits)
REDUCED = [(9, 64, 32, 32, 1), (11, 96, 96, 32, 1), (23, 320, 320, 32, 2), (32, 1120, 96, 32, 7),
           (33, 96, 96, 64, 1), (50, 320, 512, 64, 2)]


@pytest.mark.parametrize("m,k,f,bm,splits", REDUCED)
def test_reduced_cases_take_the_tiles_they_name(m, k, f, bm, splits):
    p = gemm_plan(m, 2 * f, k, SWIGLU)
    assert (p.few_rows, tile(p), p.splits, p.direct) == (False, (bm, 128), splits, False)


@pytest.mark.gpu
@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("m,k,f,bm,splits", REDUCED)
def test_swiglu_in_the_slab_reduce(split, m, k, f, bm, splits):
    kernels.test_gemm_swiglu_matches_fp64(split, m, k, f)


# Past 64 rows: (m, k, f, tile, column blocks left over by the 8 XCDs)
FUSED = [(100, 256, 512, (64, 256), 4),
         (130, 200, 96, (64, 256), 1),
         (700, 320, 2080, (64, 256), 1),     # 11 row blocks
         (1009, 320, 2848, (128, 256), 7),   # 8 waves of 64 x 64
         (401, 1024, 5664, (128, 256), 5),
         (777, 256, 10272, (192, 256), 1),
         (1009, 320, 5664, (256, 256), 5),
         (997, 2048, 5632, (256, 256), 4),   # a 997-row TinyLlama prompt's gate / up
         (600, 64, 50016, (128, 512), 4),
         (1100, 320, 14336, (128, 512), 0)]


@pytest.mark.parametrize("m,k,f,shape,left", FUSED)
def test_fused_cases_take_the_tiles_they_name(m, k, f, shape, left):
    p = gemm_plan(m, 2 * f, k, SWIGLU)
    assert (tile(p), p.splits, p.direct, p.col_blocks % 8) == (shape, 1, True, left)


@pytest.mark.gpu
@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("m,k,f,shape,left", FUSED)
def test_fused_swiglu_tiles(split, m, k, f, shape, left):
    """Rows and columns that end inside a tile; (column block, split) pairs
    left over by the 8 XCDs, whose row blocks go round all of them."""
    kernels.test_gemm_swiglu_matches_fp64(split, m, k, f)


# (m, k, n, tile, splits, pairs left over by 8)
STORED = [(300, 128, 64, (64, 256), 1, 1),
          (700, 512, 4100, (64, 256), 1, 1),
          (389, 4096, 1000, (64, 256), 8, 0),
          (300, 4096, 1024, (64, 256), 10, 0),    # the last split shorter
          (260, 4096, 512, (64, 256), 13, 2),
          (261, 8192, 250, (64, 256), 16, 0),
          (997, 2048, 2560, (128, 256), 3, 6),    # a 997-row TinyLlama prompt's QKV
          (1009, 2048, 2500, (128, 256), 3, 6),
          (2100, 512, 2050, (128, 256), 1, 1),
          (1200, 1000, 8100, (192, 256), 1, 0),
          (1009, 320, 11300, (256, 256), 1, 5),
          (600, 256, 20000, (128, 512), 1, 0)]


@pytest.mark.parametrize("m,k,n,shape,splits,left", STORED)
def test_stored_cases_take_the_tiles_they_name(m, k, n, shape, splits, left):
    p = gemm_plan(m, n, k, STORE, False)  # as zr_gemm's
    assert (tile(p), p.splits, p.col_blocks * p.splits % 8) == (shape, splits, left)


@pytest.mark.gpu
@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("m,k,n,shape,splits,left", STORED)
def test_store_tiles(split, m, k, n, shape, splits, left):
    kernels.test_gemm_matches_fp64(split, m, k, n)


# Microbatches beside other streams take no more CU time than 128 x 256 tiles
# (128 x 512 ones that fill two passes) would, whatever fills a pass better.
# (rows, k, n, epilogue, tile and splits of a waiting call, of an asynchronous one)
BESIDE = [(200, 2048, 11264, SWIGLU, ((64, 256), 1), ((128, 256), 1)),
          (256, 4096, 14336, SWIGLU, ((64, 256), 1), ((128, 256), 1)),
          (600, 4096, 28672, SWIGLU, ((192, 256), 1), ((128, 256), 1)),
          (640, 4096, 14336, SWIGLU, ((192, 256), 1), ((128, 512), 1)),
          (1400, 4096, 28672, SWIGLU, ((128, 256), 1), ((128, 512), 1)),
          (997, 2048, 11264, SWIGLU, ((256, 256), 1), ((256, 256), 1)),
          (700, 4096, 6144, STORE, ((192, 256), 2), ((128, 256), 1)),
          (2108, 2048, 2048, STORE, ((192, 256), 2), ((128, 256), 1)),
          (997, 2048, 2560, STORE, ((128, 256), 3), ((128, 256), 3)),
          (208, 4096, 3072, STORE, ((128, 256), 10), ((128, 256), 10))]  # up to 256 rows: one plan


@pytest.mark.parametrize("m,k,n,epilogue,alone,beside", BESIDE)
def test_asynchronous_microbatches_take_tiles_by_their_cu_time(m, k, n, epilogue, alone, beside):
    plans = [gemm_plan(m, n, k, epilogue, w) for w in (True, False)]
    assert [(tile(p), p.splits) for p in plans] == [alone, beside]
    if beside[1] == 1:
        work = {(128, 256): 0.863, (192, 256): 1.232, (256, 256): 1.564, (64, 256): 0.493, (128, 512): 1.62}
        blocks = -(-m // 128) * -(-n // 256)
        assert plans[1].row_blocks * plans[1].col_blocks * work[beside[0]] <= 1.03 * blocks * work[128, 256]


def both_ways(cfg, lens, chunks, seed, kv_dtype="bf16"):
    """Logits of one microbatch through zr_forward and through zr_forward_staged_async."""
    geo = geometry(cfg)
    ctx, _ = make(cfg, geo, random_weights(cfg, geo, seed=5), kv_dtype, True, max_tokens=1000, max_seqs=len(chunks),
                  pages=sum((n + c + 15) // 16 + 1 for n, c in zip(lens, chunks)) * 2, pps=80)
    rng = np.random.default_rng(seed)
    toks = [rng.integers(0, cfg["vocab"], c).astype(np.uint32) for c in chunks]
    groups = ([], [])
    for n in lens:
        kv = [rng.standard_normal((cfg["num_layers"], n, geo["kv_cols"]), dtype=np.float32) for _ in range(2)]
        for g in groups:
            g.append(ctx.new_backend(2048))
            if n:
                g[-1].import_kv_cache(KVCacheSnapshot(n, n, *kv))
    _, waited = BackendMicrobatchExecutor.forward_mixed(groups[0], [t.tolist() for t in toks])
    st = stage_mixed(ctx, groups[1], chunks, np.concatenate(toks))
    S, V = len(chunks), cfg["vocab"]
    d_ids, d_logits = DeviceBuffer(ctx, 4 * S), DeviceBuffer(ctx, 4 * S * V)
    ctx.check(ctx.lib.zr_forward_staged_async(ctx.h, st, None, d_ids.ptr, d_logits.ptr))
    ctx.check(ctx.lib.zr_synchronize(ctx.h))
    got = d_logits.download(np.float32, (S, V))
    ctx.lib.zr_staged_destroy(st)
    ctx.close()
    return waited, got


MODEL = dict(hidden=256, num_heads=4, num_kv_heads=2, num_layers=2, vocab=300, ffn=7168, rms_norm_eps=1e-5,
             rope_base=10000.0)


@pytest.mark.gpu
@pytest.mark.parametrize("sessions", [0, 200, 700])
def test_waiting_and_asynchronous_calls_agree_bit_for_bit(sessions):
    """Gate / up takes other tiles, whose sums are the same, and a decode step
    (any row count) or a chunk of up to 256 rows keeps the rest of its plans."""
    rows = sessions or 200
    assert len({tile(gemm_plan(rows, 2 * MODEL["ffn"], MODEL["hidden"], SWIGLU, w)) for w in (True, False)}) == 2
    chunks = [1] * sessions or [rows]
    waited, got = both_ways(MODEL, [7] * len(chunks) if sessions else [0], chunks, rows)
    np.testing.assert_array_equal(got, waited)


@pytest.mark.gpu
def test_longer_chunks_agree_but_for_the_order_of_sums():
    """Past 256 rows a waiting chunk's other products may split K another way."""
    cfg = dict(MODEL, hidden=4096, num_heads=32, num_kv_heads=8, num_layers=1, ffn=256)
    assert [gemm_plan(700, 6144, 4096, STORE, w).splits for w in (True, False)] == [2, 1]
    waited, got = both_ways(cfg, [0], [700], 700, "f32")  # (bf16 K / V rows near a tie would round apart)
    # operands carry 2^-16 of their value, which sums in another order may round the other way: four products
    # and the head
    assert np.isfinite(got).all()
    assert np.abs(got - waited).max() <= 5 * 2.0 ** -16 * np.abs(waited).max()
