"""Rotation and append of a long prompt against the rotation written out in 64 bits: keys and values of the first layer at every position, in one
pass and in passes that start and end inside slabs of eight positions."""
import numpy as np
import pytest

from test_gpu_decoder import CFG, _build

pytestmark = pytest.mark.gpu

U16, U32 = 2.0 ** -11, 2.0 ** -24  # half an ulp


@pytest.mark.parametrize("hd,nh,nkv,n_prompt,theta", [(128, 16, 16, 1100, 1e4), (64, 24, 8, 1030, 1e6), (96, 8, 8, 1029, 1e4), (32, 4, 1, 300, 1e4)])
@pytest.mark.parametrize("rows", [None, 67])
def test_keys_and_values_of_the_first_layer(hd, nh, nkv, n_prompt, theta, rows):
    check(dict(n_heads=nh, n_kv_heads=nkv, head_dim=hd, d_model=256, rope_theta=theta), n_prompt, rows)


def check(shape, n_prompt, rows=None):
    cfg = {**CFG, **shape, "max_batch": 1, "max_ctx": 1280}
    hd, nkv, theta = cfg["head_dim"], cfg["n_kv_heads"], cfg["rope_theta"]
    rng = np.random.default_rng(hd + n_prompt)
    dec, ref = _build(rng, cfg, symmetric=True)
    prompt = rng.integers(0, cfg["vocab"], n_prompt).astype(np.int32)
    if rows:
        dec.set_prefill_rows(rows)
    dec.prefill(prompt)
    got_k, got_v = (a[0].astype(np.float64) for a in dec.get_kv(0, 1, 0, n_prompt))
    dec.close()

    h = ref.emb[prompt].astype(np.float64)
    xn = h / np.sqrt((h * h).mean(-1, keepdims=True) + cfg["rms_eps"]) * ref.norms[(0, "attn")].astype(np.float64)

    def projected(kind):
        """(values [position][head][channel], how far off a correct implementation may be): activations, weights with their scale and
        the result in fp16 each, the products added in f32 one by one"""
        w = ref.w[(0, kind)].astype(np.float64)
        y, size = xn @ w.T, np.abs(xn) @ np.abs(w).T
        e = (2.1 * U16 + (cfg["d_model"] + 44) * U32) * size
        return y.reshape(n_prompt, nkv, hd), (e + U16 * (np.abs(y) + e)).reshape(n_prompt, nkv, hd)

    v, ev = projected("v")
    assert (np.abs(got_v - v) <= ev + 2.0 ** -25).all()
    k, ek = projected("k")
    half = hd // 2
    angle = np.arange(n_prompt)[:, None] * theta ** (-2.0 * np.arange(half) / hd)  # in f32: exponent, power, reciprocal, product
    cs, sn = np.cos(angle)[:, None, :], np.sin(angle)[:, None, :]
    a, b, both = k[..., :half], k[..., half:], np.abs(k[..., :half]) + np.abs(k[..., half:])
    e = ek[..., :half] + ek[..., half:] + (both + ek[..., :half] + ek[..., half:]) * (((np.log(theta) + 10) * angle[:, None, :] + 8) * U32 + U16) + 2.0 ** -25
    assert (np.abs(got_k[..., :half] - (a * cs - b * sn)) <= e).all()
    assert (np.abs(got_k[..., half:] - (a * sn + b * cs)) <= e).all()
    # the bound tells one position, pair or head from the next: on most values it is far below what is left of a wrong angle
    assert np.median(e) < 0.05 * np.median(both) * (cfg["d_model"] / 256) ** 0.5
