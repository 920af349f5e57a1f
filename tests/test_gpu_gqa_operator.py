"""GroupQueryAttention on f32 tensors across the forms of its kernel: rows per workgroup from 16 to 256, key groups merged
through LDS, keys split over the grid, ragged ends of rows and keys, every head width; and RMSNorm at the widths where
its register form ends.  Reference: the same in float32 / float64 torch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _reference(q, k, v, hq, hkv):
    import torch

    B, Sq, _ = q.shape
    Sk = k.shape[1]
    d = q.shape[2] // hq
    qh = q.view(B, Sq, hq, d).permute(0, 2, 1, 3).contiguous()
    kh = k.view(B, Sk, hkv, d).permute(0, 2, 3, 1).repeat_interleave(hq // hkv, 1).contiguous()
    vh = v.view(B, Sk, hkv, d).permute(0, 2, 1, 3).repeat_interleave(hq // hkv, 1).contiguous()
    p = torch.softmax(torch.matmul(qh, kh) / np.sqrt(d), -1)
    return torch.matmul(p, vh).permute(0, 2, 1, 3).reshape(B, Sq, hq * d)


@pytest.mark.parametrize("B,Sq,Sk,hq,hkv,d", [
    (1, 1, 1, 4, 4, 128),         # one key
    (1, 1, 2048, 32, 8, 128),     # decode: keys split over the grid
    (2, 1, 777, 16, 2, 64),       # decode, ragged keys, eight query heads per kv head
    (4, 1, 255, 8, 8, 32),        # decode below the split
    (1, 3, 1025, 6, 2, 96),
    (1, 512, 512, 32, 8, 128),    # 64 rows per workgroup
    (2, 300, 333, 32, 8, 64),     # 64 rows, ragged
    (2, 515, 97, 32, 8, 128),     # 128 rows per workgroup
    (4, 520, 140, 32, 8, 32),     # 256 rows per workgroup, the last one part full
    (4, 512, 33, 32, 8, 96),
    (1, 17, 31, 2, 1, 128),
    # keys and values prepared in front: 64, 128 and 256 rows, ragged rows and keys, keys split over the grid
    (1, 512, 511, 32, 8, 128), (4, 300, 515, 8, 8, 32), (2, 130, 1999, 8, 2, 96), (1, 200, 2000, 32, 8, 128), (1, 90, 1290, 16, 2, 64),
    (1, 1000, 1111, 32, 8, 128), (1, 1024, 1025, 32, 8, 64), (2, 515, 1201, 32, 8, 96), (1, 1023, 1500, 32, 8, 32),
    (4, 1000, 1111, 32, 8, 64), (4, 520, 1057, 32, 8, 128), (4, 513, 800, 32, 8, 96), (4, 600, 300, 32, 8, 32),
])
def test_operator_against_float32(B, Sq, Sk, hq, hkv, d):
    import torch

    from yscv_amd import onnx_ops as ops

    g = torch.Generator(device="cuda").manual_seed(B * 1000 + Sq + Sk)
    q = torch.randn(B, Sq, hq * d, generator=g, device="cuda")
    k = torch.randn(B, Sk, hkv * d, generator=g, device="cuda")
    v = torch.randn(B, Sk, hkv * d, generator=g, device="cuda")
    got = ops.exec_grouped_query_attention(q, k, v, hq, hkv)
    want = _reference(q, k, v, hq, hkv)
    assert float((got - want).norm() / want.norm()) < 1e-3
    assert float((got - want).abs().max()) <= 4e-3 * float(want.abs().max())
    assert torch.equal(got, ops.exec_grouped_query_attention(q, k, v, hq, hkv))


@pytest.mark.parametrize("B,Sq,hq,hkv", [
    (1, (1 << 24) - 1, 2, 1),   # more rows per kv head than one launch takes: the second one starts inside the sequence
    (65535, 1, 130, 130),       # more (sequence, kv head) problems than one launch takes
])
def test_more_rows_or_problems_than_one_launch_takes(B, Sq, hq, hkv):
    import torch

    from yscv_amd import onnx_ops as ops

    q = torch.randn(B, Sq, hq * 32, device="cuda")
    k = torch.randn(B, 1, hkv * 32, device="cuda")
    # one key: the result is its value (rounded to fp16) over the softmax sum, one weight: 2^(s - round(s)) in f32, where
    # |s| is below 16 (32 channels ~N(0, 1), scaled), so 1 up to 16 * 2^-24, and one more rounding
    v = torch.randn(B, 1, hkv * 32, device="cuda").half().float()
    got = ops.exec_grouped_query_attention(q, k, v, hq, hkv)
    want = v.view(B, 1, hkv, 1, 32).expand(B, 1, hkv, hq // hkv, 32).reshape(B, 1, hq * 32)
    assert bool(((got - want).abs() <= 17 * 2.0**-24 * want.abs()).all())


@pytest.mark.parametrize("sq,sk", [(40, 50), (600, 1300)])
def test_values_on_four_byte_alignment(sq, sk):
    import torch

    from yscv_amd import onnx_ops as ops

    q, k = torch.randn(1, sq, 8 * 64, device="cuda"), torch.randn(1, sk, 2 * 64, device="cuda")
    buf = torch.randn(sk * 128 + 1, device="cuda")
    v = buf[1:].view(1, sk, 128)
    want = ops.exec_grouped_query_attention(q, k, v.clone(), 8, 2)
    assert torch.equal(ops.exec_grouped_query_attention(q, k, v, 8, 2), want)


@pytest.mark.parametrize("rows,d", [(1, 4), (3, 1022), (5, 1024), (2, 8192), (2, 8196), (70, 4096), (1, 7)])
def test_rms_norm_widths(rows, d):
    import torch

    from yscv_amd import onnx_ops as ops

    x, gamma = torch.randn(rows, d, device="cuda") * 3, torch.rand(d, device="cuda") + 0.5
    want = x.double() / torch.sqrt(x.double().square().mean(-1, keepdim=True) + 1e-5) * gamma.double()
    got = ops.rms_norm(x, gamma, 1e-5)
    assert float((got.double() - want).abs().max() / want.abs().max()) < 1e-6
    odd = torch.empty(rows * d + 1, device="cuda")
    odd[1:] = x.reshape(-1)
    assert float((ops.rms_norm(odd[1:].view(rows, d), gamma, 1e-5).double() - want).abs().max() / want.abs().max()) < 1e-6


def test_rms_norm_of_more_rows_than_one_launch_takes():
    import torch

    from yscv_amd import onnx_ops as ops

    x, gamma = torch.randn((1 << 24) + 5, 4, device="cuda"), torch.rand(4, device="cuda") + 0.5
    want = x / torch.sqrt(x.square().mean(-1, keepdim=True) + 1e-5) * gamma
    assert float((ops.rms_norm(x, gamma, 1e-5) - want).abs().max()) < 1e-5  # f32 against f32, |want| up to 3
