"""The bound that attention kernels are held to (gpu_util.attention_bound): met by fp16 weights and outputs, broken by one marked position
lost or counted twice, whatever the size of q."""
import math

import numpy as np
import pytest
from gpu_util import attention_bound, mark_block_edges, without_key


@pytest.mark.parametrize("pos", [33, 512, 1100, 2170, 4200])
@pytest.mark.parametrize("rms", [0.05, 0.3, 1.0])
def test_one_lost_position_breaks_it(pos, rms):
    rng = np.random.default_rng(pos)
    hd = 64
    q = rng.standard_normal((2, hd)) * rms
    k = (rng.standard_normal((1, pos + 1, 1, hd)) * 0.25).astype(np.float16)
    v = rng.standard_normal((1, pos + 1, 1, hd)).astype(np.float16)
    mark_block_edges(k, v)
    k, v = k[0, :, 0].astype(np.float64), v[0, :, 0].astype(np.float64)
    s = q @ k.T / math.sqrt(hd)
    p = np.exp(s - s.max(-1, keepdims=True))
    want = p @ v / p.sum(-1)[..., None]
    bound = attention_bound(p, v, want, 2.0 ** -20)
    got = (p.astype(np.float16).astype(np.float64) @ v / p.sum(-1)[..., None]).astype(np.float16)
    assert (np.abs(got - want) <= bound).all()
    for i in range(pos):
        if i % 32 in (0, 31):
            lost, total = without_key(p, v, want, i), p.sum(-1)[..., None]
            twice = (want * total + p[:, i:i + 1] * v[i]) / (total + p[:, i:i + 1])
            for wrong in (lost, twice):
                assert (np.abs(wrong - want) > 2 * bound)[:, i // 32 % hd].all(), i
