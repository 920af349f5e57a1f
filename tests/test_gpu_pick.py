"""The greedy pick and the logits that sampling looks at, at the ends of their chunks of 1024 and among ties."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _decoder(vocab, distinct, gain=1.0, **over):
    """LM head rows repeat every `distinct` rows: that many different logits, each several times."""
    from yscv_amd.decoder import Decoder

    cfg = dict(n_layers=1, d_model=128, n_heads=2, n_kv_heads=1, head_dim=64, d_ff=128, vocab=vocab, group_size=32, max_batch=3,
               max_ctx=128, max_steps=64, rope_theta=10000.0, rms_eps=1e-5)
    cfg.update(over)
    dec = Decoder(**cfg)
    dec.init_random(seed=vocab, nibbles=(1, 15))
    rng = np.random.default_rng(vocab + distinct)
    at = np.arange(vocab) % distinct
    packed = rng.integers(0, 256, (distinct, 64), dtype=np.uint8)[at]
    scales = rng.uniform(0.01, 0.02, (distinct, 4)).astype(np.float16)[at]
    dec.set_linear(0, "lm_head", packed.reshape(-1), scales.reshape(-1), vocab, 128)
    dec.set_norm(0, "final", np.full(128, gain, np.float32))
    dec.finalize()
    return dec


@pytest.mark.parametrize("vocab,distinct", [(5, 5), (1023, 7), (1024, 1), (1025, 1025), (1027, 3), (2049, 2048), (70000, 11)])
def test_the_last_of_equal_maxima(vocab, distinct):
    dec = _decoder(vocab, distinct)
    for kw in (dict(use_graph=True), dict(use_graph=False)):
        dec.reset(np.array([1, 2, 4], np.int32), 0)
        dec.run(3, **kw)
        rows, last = dec.logits(), dec.tokens(2, 1)[0]
        for b in range(3):
            assert last[b] == np.flatnonzero(rows[b] == rows[b].max())[-1]


def test_a_nan_restarts_the_scan():
    """max_by with partial_cmp or Equal: behind the last NaN the scan starts again; all logits NaN gives the last index."""
    dec = _decoder(2050, 9, gain=np.nan)
    dec.reset(np.array([1], np.int32), 0)
    dec.run(1, use_graph=True)
    assert np.isnan(dec.logits()).all() and dec.tokens(0, 1)[0, 0] == 2049


@pytest.mark.parametrize("vocab,distinct,kw", [
    (60000, 60000, dict()), (60000, 60000, dict(top_k=1)), (60000, 60000, dict(temperature=0.01)), (60000, 60000, dict(top_k=59, top_p=1.0)),
    (60000, 60000, dict(top_k=60)), (60001, 13, dict(top_p=0.5)), (60001, 4099, dict(temperature=1.7)), (1500, 1500, dict(top_k=2)),
    (60000, 60000, dict(repetition_penalty=1.2)), (60000, 60000, dict(temperature=1e-39))])
def test_generate_draws_what_the_whole_row_gives(vocab, distinct, kw):
    from yscv_amd import kernels as K

    dec = _decoder(vocab, distinct, gain=8.0)
    prompt = [1, 3, 2]
    got = dec.generate(prompt, max_tokens=10, **kw)
    opt = dict(temperature=1.0, top_k=50, top_p=0.9, repetition_penalty=1.0)
    opt.update(kw)
    state, tokens = 0xDEADBEEF, list(prompt)
    dec.prefill(np.array(prompt, np.int32))
    for g in range(10):
        row = dec.logits()[0].copy()
        if opt["repetition_penalty"] != 1.0:
            rp = np.float32(opt["repetition_penalty"])
            for t in tokens:
                row[t] = row[t] / rp if row[t] > 0 else row[t] * rp
        if opt["temperature"] != 1.0:
            with np.errstate(over="ignore", invalid="ignore", divide="ignore"):
                row = row * (np.float32(1.0) / np.float32(opt["temperature"]))
        tok, state = K.sample_token(row, opt["top_k"], opt["top_p"], state)
        assert got[g] == tok, g
        tokens.append(int(tok))
        dec.reset(np.array([tok], np.int32), len(tokens) - 1)
        dec.run(1, auto=True)


def test_generate_with_nan_logits():
    dec = _decoder(60000, 60000, gain=np.nan)
    a = dec.generate([1, 2], max_tokens=3)
    assert len(a) == 3 and (a < 60000).all()
