"""int4 matmul in tiles of 256 x 256 (many rows, enough columns to fill the CUs): ragged rows and columns, every group size
and scale type, K that ends inside a 128-k tile, column ranges split over two launches.

The kernel multiplies fp16 activations with fp16((q - zp) * scale) and adds in f32, so against those operands in 64 bits an
element may be off by at most K roundings of 2^-24 each (and one of the output) of the sum of its products' magnitudes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (m, n, k, group, scales, zero points): one round of 256 CUs is 32768 columns at 257 .. 512 rows, 16384 at 513 .. 1024 rows
CASES = [
    (257, 32768, 128, 128, "f16", False), (300, 32761, 192, 64, "f16", True), (512, 32700, 96, 32, "f16", False),
    (511, 32768, 320, 32, "f32", True), (600, 16384, 64, 64, "f32", False), (1000, 16383, 256, 256, "f16", True),
    (520, 33000, 160, 32, "f16", True), (1024, 20000, 384, 128, "f32", True), (2048, 8192, 1024, 64, "f16", False),
    # tiles of 224 and 192 columns: one round is 28672 / 24576 columns at two row tiles, 14336 / 12288 at four
    (512, 28672, 128, 128, "f16", False), (300, 28661, 192, 64, "f16", True), (1000, 14330, 320, 32, "f16", False),
    (513, 14300, 256, 128, "f32", True), (700, 14336, 160, 32, "f16", True),
    (512, 24576, 128, 128, "f16", True), (257, 24561, 192, 64, "f32", False), (1024, 12280, 320, 32, "f16", True),
    (2048, 6144, 192, 32, "f16", False),
]


@pytest.mark.parametrize("m,n,k,g,sdt,zp", CASES)
@pytest.mark.parametrize("out", ["f32", "f16"])
def test_against_64_bits(m, n, k, g, sdt, zp, out):
    import torch

    from yscv_amd import kernels as K

    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    groups = k // g
    b = torch.randint(0, 256, (n, k // 2), generator=gen, device="cuda", dtype=torch.uint8)
    sc = (torch.rand(n, groups, generator=gen, device="cuda") * 0.015 + 0.005).to(torch.float16 if sdt == "f16" else torch.float32)
    z = torch.randint(0, 16, (n, (groups + 1) // 2 * 2), generator=gen, device="cuda", dtype=torch.uint8) if zp else None
    zpk = (z[:, 0::2] | (z[:, 1::2] << 4)).reshape(-1).cpu().numpy() if zp else None
    w = K.PackedInt4Weight(b.reshape(-1).cpu().numpy(), sc.reshape(-1).cpu().numpy(), g, n, k, zero_points=zpk, nibble_format=K.NIBBLE_UNSIGNED)
    x = torch.randn(m, k, generator=gen, device="cuda").half()
    y = w.matmul(x, out_dtype=torch.float32 if out == "f32" else torch.float16)
    q = torch.stack((b & 15, b >> 4), dim=2).reshape(n, k).float()
    zf = z[:, :groups].float().repeat_interleave(g, dim=1) if zp else 8.0
    wf = ((q - zf).half() * sc.half().repeat_interleave(g, dim=1)).double()
    xd = x.double()
    off = 2.0 ** -23 if out == "f32" else 2.0 ** -11
    for c0 in range(0, n, 8192):
        want = xd @ wf[c0:c0 + 8192].t().contiguous()
        mag = xd.abs() @ wf[c0:c0 + 8192].abs().t().contiguous()
        err = (y[:, c0:c0 + 8192].double() - want).abs()
        assert bool((err <= mag * (k * 2.0 ** -24) + want.abs() * off + 1e-7).all()), c0
