"""Attention of long prompts: 32 queries per wave (a pass that fills the CUs with them) against 16 (the same prompt in shorter passes,
which the oracle's tests cover), and the long pass against a float64 causal softmax.  The second layer's cache rows depend on the first
layer's attention at their position."""
import math

import numpy as np
import pytest
from gpu_util import attention_bound, without_key

from test_gpu_decoder import CFG, _build

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,nh,nkv,n_prompt", [(32, 32, 8, 1061), (64, 32, 8, 1056), (96, 24, 6, 1400), (128, 32, 8, 1025)])
def test_one_pass_against_several(hd, nh, nkv, n_prompt):
    """(two fp16 pipelines that round alike but for the attention, behind a layer's projections; the test below is the one of the kernel)"""
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


MARKED = (0, 15, 16, 31, 32, 63, 64, 95, 96, 127, 128, 511, 512, 639, 640, 895)  # keys at the edges of row tiles and of both groups' halves of a stage


@pytest.mark.parametrize("hd,nh,nkv,n_prompt,rows", [
    (32, 32, 8, 1061, 0), (64, 32, 8, 1056, 0), (96, 24, 6, 1400, 0), (128, 32, 8, 1025, 0), (64, 16, 2, 700, 0), (128, 16, 8, 333, 0), (128, 16, 16, 130, 0),
    (64, 32, 8, 1056, 333)])  # (the last one in several passes)
def test_against_float64(hd, nh, nkv, n_prompt, rows):
    """A model that shows its first layer's attention: its output projection is the identity, its FFN zero, and the second layer's V
    projection takes one channel each out of the normalised residual.  The q heads of a group are its k head times a power of two, so
    rotated q is in the cache, too; values are large at the marked keys, in a channel of their own each."""
    from yscv_amd.decoder import Decoder

    group, d, kvd, vocab, g = nh // nkv, nh * hd, nkv * hd, 2048, 32
    rng = np.random.default_rng(nh * hd + n_prompt)
    dec = Decoder(n_layers=2, d_model=d, n_heads=nh, n_kv_heads=nkv, head_dim=hd, d_ff=128, vocab=vocab, group_size=g, max_batch=1,
                  max_ctx=(n_prompt + 135) // 128 * 128, max_steps=8, rope_theta=10000.0, rms_eps=1e-5)

    def linear(layer, kind, q, scales):  # q [n][k]: values -8 .. 7
        nib = (q + 8).astype(np.uint8)
        dec.set_linear(layer, kind, (nib[:, 0::2] | (nib[:, 1::2] << 4)).reshape(-1), scales.astype(np.float16).reshape(-1), *q.shape)

    def zero(layer, kind, n, k):
        linear(layer, kind, np.zeros((n, k), np.int8), np.full((n, k // g), 0.01))

    # keys from the lower channels of the embedding only, values from the upper ones too: the marked tokens are one-hot there
    wk = rng.integers(-7, 8, (kvd, d)).astype(np.int8)
    wk[:, d // 2:] = 0
    ks = rng.uniform(0.5, 1.5, (kvd, d // g)) * 0.2 / math.sqrt(d)
    wv = rng.integers(-7, 8, (kvd, d)).astype(np.int8)
    wv[:, d // 2:] = 0
    vs = np.full((kvd, d // g), 0.25 / math.sqrt(d))
    chan = np.arange(kvd) % hd
    special = {pos: 100 + i for i, pos in enumerate(m for m in MARKED if m < n_prompt)}
    for i in range(len(special)):  # a group of its own for each: seven times the scale in the channels of one residue
        at = d // 2 + g * (i % (d // 2 // g))
        wv[chan % len(special) == i, at + i % g] = 7
        vs[:, at // g] = 16.0 / (7 * math.sqrt(d / 2))
    linear(0, "k", wk, ks)
    linear(0, "v", wv, vs)
    head = np.arange(d) // hd
    kv_row = head // group * hd + np.arange(d) % hd
    linear(0, "q", wk[kv_row], ks[kv_row] * 2.0 ** -(head % group)[:, None])
    eye = np.zeros((d, d), np.int8)
    eye[np.arange(d), np.arange(d)] = 1
    linear(0, "o", eye, np.ones((d, d // g)))
    pick = (np.arange(kvd) // hd * group + np.arange(kvd) % group) * hd + chan  # column j of layer 1's V: this channel of the residual
    sel = np.zeros((kvd, d), np.int8)
    sel[np.arange(kvd), pick] = 1
    linear(1, "v", sel, np.ones((kvd, d // g)))
    for layer in (0, 1):
        if layer:
            zero(1, "q", d, d), zero(1, "k", kvd, d), zero(1, "o", d, d)
        zero(layer, "gate", 128, d), zero(layer, "up", 128, d), zero(layer, "down", d, 128)
        for kind in ("attn", "ffn"):
            dec.set_norm(layer, kind, np.ones(d, np.float32))
    zero(0, "lm_head", vocab, d)
    dec.set_norm(0, "final", np.ones(d, np.float32))
    emb = rng.standard_normal((vocab, d)) * 0.25
    emb[:, d // 2:] = 0
    for i, tok in enumerate(special.values()):
        emb[tok] *= 0.02
        emb[tok, d // 2 + g * (i % (d // 2 // g)) + i % g] = 0.25 * math.sqrt(d / 2)
    emb = emb.astype(np.float16)
    dec.set_embedding(emb)
    dec.finalize()
    prompt = rng.integers(200, vocab, n_prompt).astype(np.int32)
    for pos, tok in special.items():
        prompt[pos] = tok
    if rows:
        dec.set_prefill_rows(rows)
    dec.prefill(prompt)
    k0, v0 = (a.astype(np.float64)[0] for a in dec.get_kv(0, 1, 0, n_prompt))  # [position][kv head][channel]
    got = dec.get_kv(1, 1, 0, n_prompt)[1].astype(np.float64)[0].reshape(n_prompt, kvd)
    dec.close()
    attn, off = np.empty((n_prompt, nh, hd)), np.empty((n_prompt, nh, hd))
    seen = np.tri(n_prompt, dtype=bool)
    shown = {pos: 0 for pos in special}
    for h in range(nh):
        kh, vh = k0[:, h // group], v0[:, h // group]
        s = np.where(seen, (kh * 2.0 ** -(h % group)) @ kh.T / math.sqrt(hd), -np.inf)
        p = np.exp(s - s.max(-1, keepdims=True))
        attn[:, h] = p @ vh / p.sum(-1)[:, None]
        # (q is rounded to fp16 like k: exact but for subnormal ones)
        score_err = hd * 2.0 ** -24 * (np.abs(kh) @ np.abs(kh).T).max() / math.sqrt(hd) + 2.0 ** -20
        off[:, h] = attention_bound(p, vh[None], attn[:, h], score_err)
        cols = np.flatnonzero((pick // hd == h))
        for pos in special:  # would its loss show in what is compared below?
            lost = np.abs(without_key(p[-1:], vh[None], attn[-1:, h], pos) - attn[-1:, h])[0, chan[cols]]
            shown[pos] += int((lost > 4 * off[-1, h][chan[cols]]).sum())
    assert min(shown.values()) > 0, shown
    resid = emb[prompt].astype(np.float64) + attn.reshape(n_prompt, d)
    rms = np.sqrt((resid ** 2).mean(-1, keepdims=True) + 1e-5)
    want = (resid / rms)[:, pick]
    # the attention's part, the normalised row and the cache row in fp16, the norm of a row that is off
    bound = (off.reshape(n_prompt, d) / rms)[:, pick] + np.abs(want) * (2 * 2.0 ** -11 + off.reshape(n_prompt, d).max(-1, keepdims=True) / rms) + 1e-6
    err = np.abs(got - want)
    assert (err <= bound).all(), (float((err / bound).max()), np.argwhere(err > bound)[:5])
