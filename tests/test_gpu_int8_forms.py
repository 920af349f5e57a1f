"""int8 GEMM in tiles of 64 x 128 and 128 x 256, the forms of the result that the operators ask for: f32 sums with the zero point in device
memory, requantised f32 carriers, requantised and dequantised values, and bytes, with infinite and NaN scales among them.  Whole numbers and
single f32 operations, so every value has to be the exact one."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# rows, columns and K that take the small tile (few k-steps) and the large one (many), odd and even counts of k-steps, columns off four
SHAPES = [(1025, 4097, 320), (1025, 4098, 1600), (1025, 4097, 1536), (2113, 8201, 128), (2113, 8203, 4160)]


def _weights(torch, m, n, k):
    from yscv_amd import onnx_ops as O

    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    b = torch.randint(-128, 128, (k, n), generator=g, device="cuda", dtype=torch.int8)
    a = torch.randint(-128, 128, (m, k), generator=g, device="cuda", dtype=torch.int8)
    a[::97] = 0  # sums of 0
    return a, b, O.PrepackedI8B(b.float())


def _sums(a, b):
    return (a.double() @ b.double()).float()  # the sums are whole numbers below 2^53; one rounding to f32


def _away(torch, v):
    t = torch.trunc(v)
    return torch.where((v - t).abs() >= 0.5, t + torch.copysign(torch.ones_like(v), v), t)


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_dynamically_quantised_sums(m, n, k):
    import torch

    from yscv_amd import onnx_ops as O

    _, b, w = _weights(torch, m, n, k)
    x = torch.randn(m, k, generator=torch.Generator(device="cuda").manual_seed(k), device="cuda")
    out, _, zp = O.exec_dql_matmul_integer(x, w)
    q = O.exec_dynamic_quantize_linear(x)[0].double()
    assert torch.equal(out, ((q - float(zp)) @ b.double()).float())
    w.close()


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("b_scale", ["spread", "inf", "nan"])
def test_requantised_carriers(m, n, k, b_scale):
    import torch

    from yscv_amd import onnx_ops as O

    a, b, w = _weights(torch, m, n, k)
    comp = {"spread": 0.008 / math.sqrt(k), "inf": math.inf, "nan": math.nan}[b_scale]
    comp32 = float(np.float32(comp))
    v = _sums(a, b) * comp32 + 3.0
    r = _away(torch, v)
    # clamp keeps a NaN (a sum of 0 times an infinite scale is one too)
    want = torch.where(torch.isnan(v), v, r.clamp(-128.0, 127.0))
    got, path = O.exec_qlinear_matmul(a.float(), 1.0, 0.0, None, comp32, 0.0, 1.0, 3.0, w)
    assert path == 0
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.nan_to_num(got, 0.25), torch.nan_to_num(want, 0.25))
    # dequantised: the byte, which is 0 for a NaN, times the scale of the result
    want = torch.where(torch.isnan(v), torch.zeros_like(v), r.clamp(-128.0, 127.0))
    got = O.exec_qdq_matmul(a.float(), 1.0, w, comp32, 1.0, 3.0)
    assert torch.equal(got, (want - 3.0) * 1.0)
    w.close()


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_bytes_of_infinite_and_nan_scales(m, n, k):
    import torch

    from yscv_amd import kernels as K

    a, b, w = _weights(torch, m, n, k)
    w.close()
    p = K.pack_i8_b_for_matmul(b.cpu().numpy(), k, n)
    comp = torch.full((n,), 0.05 / math.sqrt(k), device="cuda")
    comp[0::5], comp[1::5], comp[2::5], comp[3::5] = math.inf, math.nan, 3e38, -math.inf
    v = _sums(a, b) * comp + 14.0
    for mode in (K.ROUND_HALF_AWAY, K.ROUND_TIES_EVEN):
        r = _away(torch, v) if mode == K.ROUND_HALF_AWAY else torch.round(v)
        want = torch.where(torch.isnan(v), torch.zeros_like(v), r.clamp(-100.0, 90.0))
        got = p.matmul_requant(a, 0, comp, 14.0, mode, -100, 90)
        assert torch.equal(got.to(torch.int32), want.to(torch.int32))
