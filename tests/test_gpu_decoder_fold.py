"""The multi-kernel decode step with its norms folded into the projections around them where K ends inside a 512-k slice (widths
that are no multiple of 512), for one row and for several, against the numpy restatement."""
import numpy as np
import pytest

from test_gpu_decoder import LOGIT_TOL, _build

pytestmark = pytest.mark.gpu

BASE = dict(n_layers=2, vocab=320, group_size=32, max_ctx=256, max_steps=16, rope_theta=10000.0, rms_eps=1e-5)
SHAPES = {
    "k2816": dict(d_model=1024, n_heads=16, n_kv_heads=2, head_dim=64, d_ff=2816),
    "k768": dict(d_model=768, n_heads=6, n_kv_heads=2, head_dim=128, d_ff=1408),
    "one_slice": dict(d_model=256, n_heads=4, n_kv_heads=4, head_dim=64, d_ff=640),  # four rows on one wave
}


@pytest.mark.parametrize("name,batch", [("k2816", 1), ("k2816", 2), ("k2816", 8), ("k768", 1), ("k768", 5), ("one_slice", 4)])
def test_steps_match_numpy(name, batch):
    rng = np.random.default_rng(8000 + batch)
    cfg = dict(BASE, **SHAPES[name], max_batch=batch)
    dec, ref = _build(rng, cfg, symmetric=True)
    tok = rng.integers(0, cfg["vocab"], batch).astype(np.int32)
    dec.reset(tok, 0)
    for step in range(4):
        dec.run(1, use_graph=bool(step & 1))
        exp, got = ref.step(tok, step), dec.logits()
        assert float(np.abs(got - exp).max() / np.abs(exp).max()) < LOGIT_TOL, step
        tok = dec.tokens(step, 1)[0].copy()


@pytest.mark.parametrize("name,batch", [("k2816", 9), ("k2816", 16), ("k768", 16), ("one_slice", 5)])
def test_more_rows_than_four_to_a_wave_grow_without_a_bound(name, batch):
    """Widths up to 1024 have two waves or fewer: such batches have their norms in f32.  An embedding far below sqrt(eps) and cached values of
    some hundred raise a row from 2^-8 (eps in it) to 2^10 within the first update, and the norm behind it multiplies by 16: past what an
    unnormalised fp16 row holds."""
    rng = np.random.default_rng(8100 + batch)
    cfg = dict(BASE, **SHAPES[name], max_batch=batch)
    dec, ref = _build(rng, cfg, symmetric=True, emb_scale=2.0 ** -13)
    shape = (batch, 40, cfg["n_kv_heads"], cfg["head_dim"])
    for layer in range(cfg["n_layers"]):
        k = rng.standard_normal(shape).astype(np.float16)
        v = np.broadcast_to((rng.choice([-1.0, 1.0], (batch, 1) + shape[2:]) * rng.uniform(512, 1024, (batch, 1) + shape[2:])), shape).astype(np.float16)
        dec.set_kv(layer, k, v)
        ref.set_kv(layer, k.astype(np.float32), v.astype(np.float32))
    ref.norms[(0, "ffn")] *= np.float32(16.0)
    dec.set_norm(0, "ffn", ref.norms[(0, "ffn")])
    dec.finalize()
    tok = rng.integers(0, cfg["vocab"], batch).astype(np.int32)
    dec.reset(tok, 40)
    dec.run(1)
    exp, got = ref.step(tok, 40), dec.logits()
    for row in range(batch):
        assert float(np.abs(got[row] - exp[row]).max() / np.abs(exp[row]).max()) < LOGIT_TOL, row
