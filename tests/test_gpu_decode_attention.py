"""Attention of a decode step over the fp16 cache (csrc/decode_attention.hip) where it can go wrong: one share, the edges of shares and of
blocks of 32, merges over several levels, more than sixteen query heads per kv head; against a float64 softmax over the cache rows and the
rotated q that the decoder itself reports."""
import math

import numpy as np
import pytest
from gpu_util import attention_bound, mark_block_edges, without_key

pytestmark = pytest.mark.gpu


def _decoder(heads, batch, max_ctx, qk_scale=None):
    from yscv_amd.decoder import Decoder

    nh, nkv, hd = heads
    dec = Decoder(n_layers=1, d_model=256, n_heads=nh, n_kv_heads=nkv, head_dim=hd, d_ff=256, vocab=512, group_size=32, max_batch=batch,
                  max_ctx=max_ctx, max_steps=8, rope_theta=10000.0, rms_eps=1e-5)
    dec.init_random(seed=3, nibbles=(1, 15))
    if qk_scale:
        rng = np.random.default_rng(5)
        for kind, n, scale in (("q", nh * hd, qk_scale), ("k", nkv * hd, qk_scale), ("v", nkv * hd, 0.0125)):
            nib = rng.integers(1, 16, (2, n * 128), dtype=np.uint8)
            dec.set_linear(0, kind, nib[0] | (nib[1] << 4), np.full(n * 8, scale, np.float16), n, 256)
    dec.finalize()
    return dec


@pytest.mark.parametrize("heads,batch,max_ctx,positions", [
    ((16, 4, 128), 16, 2176, (0, 31, 32, 511, 512, 1023, 1024, 1100, 2170)),  # 64 pairs: up to four shares
    ((32, 8, 128), 16, 2176, (511, 512, 2100)),                               # two shares, the 7B head layout
    ((16, 2, 64), 3, 4224, (5, 512, 700, 1600, 4200)),                        # eight shares
    ((36, 2, 32), 2, 1152, (40, 600, 1150)),                                  # eighteen query heads per kv head: two blocks of them
    ((12, 4, 96), 5, 1152, (63, 1025)),
], ids=["16q4kv-hd128", "32q8kv-hd128", "16q2kv-hd64", "36q2kv-hd32", "12q4kv-hd96"])
def test_against_float64(heads, batch, max_ctx, positions):
    nh, nkv, hd = heads
    dec = _decoder(heads, batch, max_ctx, qk_scale=0.5 / 70)  # (q and the token's key of rms 1/2: no key takes all the weight)
    rng = np.random.default_rng(17)
    k = (rng.standard_normal((batch, max_ctx - 8, nkv, hd)) * 0.5).astype(np.float16)
    v = rng.standard_normal((batch, max_ctx - 8, nkv, hd)).astype(np.float16)
    mark_block_edges(k, v)
    tokens = (np.arange(batch) * 7 + 3).astype(np.int32)
    for pos in positions:
        kp, vp = k.copy(), v.copy()
        kp[:, pos:], vp[:, pos:] = np.nan, np.nan  # what lies behind the context must not be seen
        dec.set_kv(0, kp, vp)
        outs = []
        for use_graph in (False, True, True):  # the slots of the merge are empty again behind every launch
            dec.reset(tokens, pos)
            dec.run(1, use_graph=use_graph)
            outs.append(dec.activation("attn_out"))
        assert np.array_equal(outs[0], outs[1]) and np.array_equal(outs[0], outs[2])
        q = dec.activation("qkv")[:, : nh * hd].reshape(batch, nkv, nh // nkv, hd).astype(np.float64)
        kc, vc = (a.astype(np.float64).transpose(0, 2, 1, 3) for a in dec.get_kv(0, batch, 0, pos + 1))
        s = q @ kc.transpose(0, 1, 3, 2) / math.sqrt(hd)
        p = np.exp(s - s.max(-1, keepdims=True))
        v4 = vc[:, :, None]
        want = (p @ vc) / p.sum(-1)[..., None]
        # a score: f32 sums of hd exact products, scaled; its exponential
        score_err = hd * 2.0 ** -24 * (np.abs(q) @ np.abs(kc.transpose(0, 1, 3, 2))).max() / math.sqrt(hd) + 2.0 ** -21
        bound = attention_bound(p, v4, want, score_err)
        err = np.abs(outs[0].reshape(want.shape) - want)
        assert (err <= bound).all(), (pos, float((err / bound).max()))
        for i in range(pos):  # and a marked position lost for a kv head would show
            if i % 32 in (0, 31):
                ch = i // 32 % hd
                lost = without_key(p, v4, want, i)
                assert (np.abs(lost - want) > 2 * bound)[..., ch].all(), (pos, i)
    dec.close()


def test_weights_of_shares_at_large_scores():
    """Every key of a share is the same row or zero, so its weights are exactly 1 or 0 and only the meeting of the shares can round: with
    values of +1 in one share and -1 in the other the result is (n0 - n1) / (n0 + n1) whatever the score, which reaches 1e5 here (a log
    of the weights' sum in f32 would be off by 2^-8 there)."""
    nh, nkv, hd = heads = (16, 2, 64)
    batch, max_ctx, pos = 3, 4224, 1024
    dec = _decoder(heads, batch, max_ctx)
    tokens = (np.arange(batch) * 7 + 3).astype(np.int32)
    dec.reset(tokens, pos)
    dec.run(1)
    q = dec.activation("qkv")[:, : nh * hd].reshape(batch, nkv, nh // nkv, hd).astype(np.float64)
    # along the first head of each kv head, of a size that brings its score to 1e5
    k0 = q[:, :, 0] / (q[:, :, 0] ** 2).sum(-1, keepdims=True) * 1e5 * math.sqrt(hd)
    assert np.abs(k0).max() < 65504
    k = np.repeat(k0.astype(np.float16)[:, None], max_ctx - 8, axis=1)
    v = np.ones_like(k)
    k[:, 300:512] = 0  # 300 keys that count against 512
    v[:, 512:1024] = -1
    dec.set_kv(0, k, v)
    for use_graph in (False, True):
        dec.reset(tokens, pos)
        dec.run(1, use_graph=use_graph)
        got = dec.activation("attn_out").reshape(batch, nkv, nh // nkv, hd).astype(np.float64)
        scores = (q * k[:, 0].astype(np.float64)[:, :, None]).sum(-1) / math.sqrt(hd)
        large = scores > 1000.0  # (the token's own key, and zero keys, have no weight there)
        assert large[:, :, 0].all()
        want = (300.0 - 512.0) / 812.0
        assert np.abs(got[large] - want).max() <= 2.0 ** -11 * abs(want) * 1.01, np.abs(got[large] - want).max()  # one rounding to fp16
    dec.close()
