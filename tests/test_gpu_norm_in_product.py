"""Steps of one or two rows normalise inside the QKV and gate / up products.

The same sessions in a step of nine rows run the norm kernel and the tiles:
their logits agree, at a width below a workgroup's first sweep of the row (256
threads of 8 columns), at one that ends inside the second and at the widest;
and with one, two (both loaded ahead) and more split-K slabs of O and down to
add to the residual stream.
"""
import numpy as np
import pytest

from mesh_amd import BackendMicrobatchExecutor, DecodeMicrobatchRequest, KVCacheSnapshot
from tests.test_gpu_gemm_tiles import STORE, SWIGLU, gemm_plan
from tests.test_gpu_model import make
from tests.testmodels import geometry, random_weights


@pytest.mark.gpu
@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("rows", [1, 2])
@pytest.mark.parametrize("heads,kv_heads,head_dim", [(17, 17, 64), (24, 8, 128), (32, 8, 128)])
def test_few_rows_equal_the_same_rows_of_a_larger_step(heads, kv_heads, head_dim, rows, split):
    compare_steps(heads, kv_heads, head_dim, 256, rows, split)


# (heads, kv heads, head dim, FFN, slabs of O, slabs of down)
SLABS = [(32, 4, 64, 5632, 2, 2), (16, 16, 64, 4096, 1, 4), (8, 2, 64, 8192, 1, 8)]


@pytest.mark.parametrize("rows", [1, 2])
@pytest.mark.parametrize("heads,kv_heads,head_dim,ffn,o,down", SLABS)
def test_slab_cases_leave_the_slabs_they_name(heads, kv_heads, head_dim, ffn, o, down, rows):
    h = heads * head_dim
    assert gemm_plan(rows, h, h, STORE).splits == o and gemm_plan(rows, h, ffn, STORE).splits == down
    # ... and both products that normalise are unsplit
    assert gemm_plan(rows, h + 2 * kv_heads * head_dim, h, STORE).direct and gemm_plan(rows, 2 * ffn, h, SWIGLU).direct


@pytest.mark.gpu
@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("rows", [1, 2])
@pytest.mark.parametrize("heads,kv_heads,head_dim,ffn,o,down", SLABS)
def test_residual_slabs(heads, kv_heads, head_dim, ffn, o, down, rows, split):
    compare_steps(heads, kv_heads, head_dim, ffn, rows, split)


def compare_steps(heads, kv_heads, head_dim, ffn, rows, split):
    cfg = dict(hidden=heads * head_dim, num_heads=heads, num_kv_heads=kv_heads, num_layers=2, vocab=512, ffn=ffn,
               rms_norm_eps=1e-5, rope_base=10000.0)
    geo = geometry(cfg)
    ctx, _ = make(cfg, geo, random_weights(cfg, geo, seed=7), "f32", split, max_tokens=16, max_seqs=16, pages=256,
                  pps=16)
    rng = np.random.default_rng(rows)
    lens = [21, 40, 1, 16, 17, 5, 60, 33, 2]
    groups = ([], [])
    for n in lens:
        kv = [rng.standard_normal((2, n, geo["kv_cols"]), dtype=np.float32) for _ in range(2)]
        for g in groups:
            g.append(ctx.new_backend(4096))
            g[-1].import_kv_cache(KVCacheSnapshot(n, n, *kv))

    def step(sessions, toks):
        reqs = [DecodeMicrobatchRequest(str(i), int(t), s) for i, (t, s) in enumerate(zip(toks, sessions))]
        return np.stack([o.logits for o in BackendMicrobatchExecutor.decode_step_batch(reqs, want_logits=True)])

    # operands carry 2^-16 (bf16: 2^-8) of their value, which sums in another
    # order may round the other way: four products a layer, two layers, the head
    tol = 9 * (2.0 ** -16 if split else 2.0 ** -8)
    for k in range(3):
        toks = rng.integers(0, cfg["vocab"], len(lens))
        few, many = step(groups[0][:rows], toks[:rows]), step(groups[1], toks)[:rows]
        assert np.isfinite(few).all()
        assert np.abs(few - many).max() <= tol * np.abs(many).max(), k
    ctx.close()
