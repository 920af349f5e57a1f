"""DynamicQuantizeLinear of several blocks: more block ranges than a workgroup has threads, one load per thread and several, values
behind the loads that go out ahead, NaN among them: scale, zero point and every value as the definition gives them in f32."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _away(v):
    return np.trunc(v) + np.where(np.abs(v - np.trunc(v)) >= np.float32(0.5), np.copysign(np.float32(1), v), np.float32(0))


# 1024 values per block up to 1024 blocks, four loads of a block's threads ahead: 2^20 values one load, 2^22 four
@pytest.mark.parametrize("n", [24580, 131072, 261 * 1024 - 4, (1 << 20) - 4, (1 << 20) + 4, (1 << 22) + 4, (1 << 22) + 3])
@pytest.mark.parametrize("kind", ["first", "last", "nan"])
def test_against_the_definition(n, kind):
    import torch

    from yscv_amd import onnx_ops as O

    x = np.random.default_rng(n).standard_normal(n).astype(np.float32)
    x[0 if kind == "first" else -1] = -90.0
    x[n // 3] = 60.0
    if kind == "nan":  # never wins; quantised to 0
        x[[1, n // 2]] = np.nan
    y, scale, zp = O.exec_dynamic_quantize_linear(torch.from_numpy(x).cuda())
    s = np.float32(np.float32(150.0) / np.float32(255))
    z = np.float32(np.clip(_away(-np.float32(np.float32(-90.0) / s)), 0, 255))
    assert float(scale.reshape(-1)[0]) == float(s) and float(zp.reshape(-1)[0]) == float(z)
    v = (x / s).astype(np.float32) + z
    want = np.where(np.isnan(v), np.float32(0), np.clip(_away(v), 0, 255)).astype(np.float32)
    assert np.array_equal(y.cpu().numpy().astype(np.float32).reshape(-1), want)
