"""DynamicQuantizeLinear of infinite values, of one workgroup and of several: the range is infinite, and scale, zero point and every value follow as the
definition gives them in f32 (NaN among them)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _away(v):
    return np.trunc(v) + np.where(np.abs(v - np.trunc(v)) >= np.float32(0.5), np.copysign(np.float32(1), v), np.float32(0))


@pytest.mark.parametrize("n", [7, 4096, 24580, 131072, (1 << 20) + 3, (1 << 22) + 4])
@pytest.mark.parametrize("kind", ["+", "-", "both"])
def test_against_the_definition(n, kind):
    import torch

    from yscv_amd import onnx_ops as O

    x = np.random.default_rng(n).standard_normal(n).astype(np.float32)
    if kind != "-":
        x[n // 2] = np.inf
    if kind != "+":
        x[-1] = -np.inf
    y, scale, zp = O.exec_dynamic_quantize_linear(torch.from_numpy(x).cuda())
    with np.errstate(invalid="ignore"):
        mn, mx = min(np.float32(0), x.min()), max(np.float32(0), x.max())
        s = np.float32(mx - mn) / np.float32(255)
        z = np.clip(_away(np.float32(0) - mn / s), 0, 255).astype(np.float32)  # keeps a NaN
        v = _away((x / s).astype(np.float32) + z)
    want = np.where(np.isnan(v), np.float32(0), np.clip(v, 0, 255)).astype(np.float32)
    assert np.array_equal(np.float32(scale.item()), s) and np.array_equal(np.float32(zp.item()), z, equal_nan=True)
    assert np.array_equal(y.cpu().numpy().reshape(-1), want)
