"""DynamicQuantizeLinear on both sides of the size up to which every workgroup takes the range itself, odd lengths, and values that decide
it at the ends: scale, zero point and every value as the definition gives them in f32."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _away(v):
    return np.trunc(v) + np.where(np.abs(v - np.trunc(v)) >= 0.5, np.sign(v), 0)


@pytest.mark.parametrize("n", [1, 3, 4, 1024, 8192, 24572, 24575, 24576, 24580, 32768])
@pytest.mark.parametrize("kind", ["normal", "positive", "first", "last", "zero"])
def test_against_the_definition(n, kind):
    import torch

    from yscv_amd import onnx_ops as O

    rng = np.random.default_rng(n)
    x = rng.standard_normal(n).astype(np.float32)
    if kind == "positive":
        x = np.abs(x) + np.float32(0.5)
    elif kind == "first":
        x[0] = -90.0
    elif kind == "last":
        x[-1] = 70.0
    elif kind == "zero":
        x[:] = 0.0
    y, scale, zp = O.exec_dynamic_quantize_linear(torch.from_numpy(x).cuda())
    mn, mx = np.minimum(x.min(), np.float32(0)), np.maximum(x.max(), np.float32(0))
    rng_ = np.float32(mx - mn)
    s = np.float32(1.0) if abs(rng_) < np.float32(1.1920929e-7) else np.float32(rng_ / np.float32(255))
    z = np.clip(_away(np.float32(0) - np.float32(mn / s)), 0, 255)
    assert float(scale.reshape(-1)[0]) == float(s) and float(zp.reshape(-1)[0]) == float(z)
    v = (x / s).astype(np.float32) + np.float32(z)
    assert np.array_equal(y.cpu().numpy().astype(np.float32).reshape(-1), np.clip(_away(v), 0, 255).astype(np.float32))
