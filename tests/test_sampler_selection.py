"""The sampler's selections (k-th largest logit, top-p prefix) at the sizes where its blocks, its heap and its sorted
prefixes end; needs no GPU.  The distribution left behind in the logits is compared with one worked out from numpy's
sorts, and infinities and NaN take the route they took before."""
import numpy as np
import pytest


def _expected(logits, top_k, top_p):
    n = logits.size
    l = logits.astype(np.float64)
    if 0 < top_k < n:
        l = np.where(logits < np.sort(logits)[::-1][top_k - 1], -np.inf, l)
    p = np.exp(l - l.max())
    p /= p.sum()
    if top_p < 1.0:
        order = np.argsort(-p, kind="stable")
        keep = int(np.searchsorted(np.cumsum(p[order]), top_p, side="right")) + 1
        cut = np.zeros(n)
        cut[order[:keep]] = p[order[:keep]]
        p = cut / cut.sum()
    return p


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 129, 3000, 20000])
@pytest.mark.parametrize("top_k", [0, 1, 50, 64, 1024, 1025, 2999])
@pytest.mark.parametrize("top_p,spread", [(1.0, 1.0), (0.9, 8.0), (0.9, 0.01), (0.5, 1.0)])
def test_kept_distribution(n, top_k, top_p, spread):
    from yscv_amd import kernels as K

    rng = np.random.default_rng(n * 7 + top_k)
    logits = (rng.permutation(n) / n * spread).astype(np.float32)  # distinct, so that no tie decides the kept set
    want = _expected(logits, top_k, top_p)
    got = logits.copy()
    tok, _ = K.sample_token(got, top_k, top_p, 0x1234567 + n)
    assert got[tok] > 0.0
    # a cumulative sum within rounding of top_p may keep one token more or less
    assert abs(int((got > 0).sum()) - int((want > 0).sum())) <= (1 if top_p < 1.0 else 0)
    assert np.abs(got - want).max() <= 2e-3 * want.max() + (want.max() if n < 3 else 2.0 / max(int((want > 0).sum()), 1) * want.max())


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
