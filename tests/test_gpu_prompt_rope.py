"""Rotation and append of a prompt whose slabs have more channels of v than a pass has threads for, against the same prompt in short passes
that start and end inside slabs: every row of the caches.  (The projections in front round to fp16 in kernels of their own.)"""
import numpy as np
import pytest

from test_gpu_decoder import CFG, _build

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,nh,nkv,n_prompt", [(128, 16, 16, 1100), (64, 24, 24, 1030), (96, 8, 8, 1029)])
def test_one_pass_against_short_ones(hd, nh, nkv, n_prompt):
    rng = np.random.default_rng(hd + n_prompt)
    cfg = dict(CFG, n_heads=nh, n_kv_heads=nkv, head_dim=hd, d_model=256, max_batch=1, max_ctx=1280)
    dec, _ = _build(rng, cfg, symmetric=True)
    prompt = rng.integers(0, cfg["vocab"], n_prompt).astype(np.int32)
    dec.prefill(prompt)
    want = dec.get_kv(0, 1, 0, n_prompt)
    dec.set_prefill_rows(67)
    dec.prefill(prompt)
    for got, exp in zip(dec.get_kv(0, 1, 0, n_prompt), want):
        exp = exp.astype(np.float32)
        assert np.abs(got.astype(np.float32) - exp).max() <= 1e-2 * np.abs(exp).max()
    dec.close()
