"""The sampler's selections (k-th largest logit, top-p prefix) at the sizes where its blocks, its heap and its sorted
prefixes end; needs no GPU.  Token and distribution are held bit by bit against sample_token as the reference writes it, on
full sorts (crates/yscv-onnx/src/generate.rs:121-208), and infinities and NaN take the route they took before."""
import ctypes

import numpy as np
import pytest

_expf = ctypes.CDLL("libm.so.6").expf
_expf.restype, _expf.argtypes = ctypes.c_float, [ctypes.c_float]


def _draw(state):
    """xorshift64 step and the f32 in [0, 1] it gives"""
    mask = (1 << 64) - 1
    state ^= (state << 13) & mask
    state ^= state >> 7
    state ^= (state << 17) & mask
    return np.float32(np.uint64(state)) / np.float32(2.0**64)


def _sorted_route(logits, top_k, top_p, u):
    """Every operation in f32 and in the reference's order (np.cumsum adds from left to right)."""
    l = logits.copy()
    n = l.size
    if 0 < top_k < n:
        l[l < l[np.argsort(-l, kind="stable")[top_k - 1]]] = -np.inf
    shifted = l - l.max()
    p = np.array([_expf(float(v)) if v > -np.inf else 0.0 for v in shifted], np.float32)
    p *= np.float32(1.0) / np.cumsum(p)[-1]
    if top_p < 1.0:
        order = np.argsort(-p, kind="stable")
        over = np.flatnonzero(np.cumsum(p[order]) > np.float32(top_p))
        if over.size:
            p[order[over[0] + 1:]] = 0.0
        total = np.cumsum(p)[-1]
        if total > 0:
            p *= np.float32(1.0) / total
    hit = np.flatnonzero(np.cumsum(p) > u)
    return (int(hit[0]) if hit.size else int(n - 1 - np.argmax(p[::-1]))), p


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 129, 3000, 20000])
@pytest.mark.parametrize("top_k", [0, 1, 50, 64, 1024, 1025, 2999])
@pytest.mark.parametrize("top_p,spread,distinct", [(1.0, 1.0, True), (0.9, 8.0, True), (0.9, 0.01, True), (0.5, 1.0, True),
                                                   (0.9, 30.0, False), (0.95, 1.0, False), (0.0, 1.0, False)])
def test_same_bits_as_the_sorted_route(n, top_k, top_p, spread, distinct):
    from yscv_amd import kernels as K

    rng = np.random.default_rng(n * 7 + top_k)
    level = rng.permutation(n) / n if distinct else rng.integers(0, 40, n) / 40  # many ties at every threshold otherwise
    logits = (level * spread).astype(np.float32)
    state = 0x1234567 + n
    want_tok, want = _sorted_route(logits, top_k, top_p, _draw(state))
    got = logits.copy()
    tok, _ = K.sample_token(got, top_k, top_p, state)
    assert tok == want_tok
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("n,top_k", [(100, 10), (5000, 50), (5000, 1500)])
def test_ties_at_the_threshold_are_all_kept_and_minus_infinity_never(n, top_k):
    from yscv_amd import kernels as K

    logits = np.zeros(n, np.float32)
    logits[::3] = 1.0
    logits[1::3] = -np.inf
    ones = logits == 1.0
    got = logits.copy()
    K.sample_token(got, top_k, 1.0, 99)
    if top_k <= ones.sum():
        assert np.array_equal(got > 0, ones)
    else:
        assert np.array_equal(got > 0, np.isfinite(logits))


def test_nan_and_infinity_still_draw_a_token():
    from yscv_amd import kernels as K

    for bad in (np.nan, np.inf):
        logits = np.linspace(-1, 1, 200).astype(np.float32)
        logits[17] = bad
        tok, _ = K.sample_token(logits, 20, 0.9, 5)
        assert 0 <= tok < 200
