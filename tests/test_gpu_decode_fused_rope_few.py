"""Steps of at most 8 sessions take RoPE + KV append inside the attention
launch at any split length; they equal the step with the separate kernel bit
for bit: greedy ids and every K / V row, over page ends and sliding windows
(the first page of a split may be the one the row is appended to)."""
import numpy as np
import pytest

from tests.test_gpu_model import SMALL, make
from tests.test_gpu_step_graph import _same_sessions, _sync_steps, _twin_sessions
from tests.testmodels import geometry, random_weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kv_dtype", ["bf16", "f32"])
@pytest.mark.parametrize("lens,windows", [([1], [4096]), ([517], [4096]),
                                          ([1, 15, 16, 17, 40, 100, 250, 60],
                                           [4096, 4096, 4096, 4096, 48, 4096, 4096, 70])])
def test_few_sessions_equal_the_separate_rope_kernel(monkeypatch, kv_dtype, lens, windows):
    cfg = SMALL
    geo = geometry(cfg)
    weights = random_weights(cfg, geo, seed=41, std=0.05)
    ctx, _ = make(cfg, geo, weights, kv_dtype, True, max_tokens=16, max_seqs=16, pages=1024, pps=64)
    rng = np.random.default_rng(41)
    a, b = _twin_sessions(ctx, rng, lens, windows, geo["kv_cols"], cfg["num_layers"])
    first = rng.integers(0, cfg["vocab"], len(lens))
    got = _sync_steps(b, first, 20, want_logits=True)
    monkeypatch.setenv("ZR_ATTN_FUSE_ROPE", "0")
    want = _sync_steps(a, first, 20, want_logits=True)
    for k in range(20):
        np.testing.assert_array_equal(got[k], want[k], err_msg=f"step {k}")
    _same_sessions(a, b)
    ctx.close()
