"""Attention of long prompts: 32 queries per wave (a pass that fills the CUs with them) against 16 (the same prompt in shorter passes,
which the oracle's tests cover).  The second layer's cache rows depend on the first layer's attention at their position; both forms round
weights and outputs to fp16, so rows agree to a few of those."""
import numpy as np
import pytest

from test_gpu_decoder import CFG, _build

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,nh,nkv,n_prompt", [(32, 32, 8, 1061), (64, 32, 8, 1056), (96, 24, 6, 1400), (128, 32, 8, 1025)])
def test_one_pass_against_several(hd, nh, nkv, n_prompt):
    rng = np.random.default_rng(hd)
    cfg = dict(CFG, n_heads=nh, n_kv_heads=nkv, head_dim=hd, d_model=256, max_batch=1, max_ctx=1536)
    dec, _ = _build(rng, cfg, symmetric=True)
    prompt = rng.integers(0, cfg["vocab"], n_prompt).astype(np.int32)
    dec.prefill(prompt)
    logits = dec.logits().copy()
    caches = [dec.get_kv(l, 1, 0, n_prompt) for l in range(cfg["n_layers"])]
    dec.set_prefill_rows(300)
    dec.prefill(prompt)
    got = dec.logits()
    assert np.abs(got - logits).max() <= 1e-2 * np.abs(logits).max()
    for l, (ek, ev) in enumerate(caches):
        gk, gv = dec.get_kv(l, 1, 0, n_prompt)
        for g, e in ((gk, ek), (gv, ev)):
            assert np.isfinite(g.astype(np.float32)).all()
            assert np.abs(g.astype(np.float32) - e.astype(np.float32)).max() <= 1e-2 * np.abs(e.astype(np.float32)).max(), l
    dec.close()
