"""int4 matmul in the tiles of the wide GEMM that a plan picks by size: 128-row tiles, K cut over workgroups, two launches, rows that
end off a vector in every output type, f32 rows (scaled by rows).

Against fp16((q - zp) * scale) and the fp16 activations in 64 bits an element may be off by at most K roundings of 2^-24 each (and one
of the output) of the sum of its products' magnitudes; f32 rows are rounded to fp16 once more, 2^-11 of each product."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# m, n, k, group, zero points
CASES = [
    (129, 24577, 192, 64, False), (150, 28672, 128, 128, True), (255, 12289, 320, 32, False),  # 128 x 192 and 128 x 256
    (700, 5632, 384, 32, True), (2048, 4096, 192, 64, False),
    (1024, 24002, 576, 64, False),                                                           # whole rounds, then the rest
    (300, 4096, 4096, 32, False), (260, 2050, 8192, 128, True), (991, 469, 7520, 32, False),  # K in parts
    (66, 50001, 96, 32, False),
    (147, 6085, 1952, 32, True), (66, 12518, 4672, 64, False),                               # K in parts: 128 x 192, 128 x 256
    (1894, 257, 3200, 128, False), (925, 203, 4640, 32, True),                               # and the LDS-ring GEMM's 128 and 64 rows
    (811, 22008, 96, 32, False), (415, 53494, 96, 32, True), (921, 21739, 192, 64, False),   # whole rounds, then the rest
]


@pytest.mark.parametrize("m,n,k,g,zp", CASES)
@pytest.mark.parametrize("act", ["f32", "f16", "bf16"])
def test_against_64_bits(m, n, k, g, zp, act):
    import torch

    from yscv_amd import kernels as K

    dt = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[act]
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    groups = k // g
    b = torch.randint(0, 256, (n, k // 2), generator=gen, device="cuda", dtype=torch.uint8)
    sc = (torch.rand(n, groups, generator=gen, device="cuda") * 0.015 + 0.005).half()
    z = torch.randint(0, 16, (n, (groups + 1) // 2 * 2), generator=gen, device="cuda", dtype=torch.uint8) if zp else None
    zpk = (z[:, 0::2] | (z[:, 1::2] << 4)).reshape(-1).cpu().numpy() if zp else None
    w = K.PackedInt4Weight(b.reshape(-1).cpu().numpy(), sc.reshape(-1).cpu().numpy(), g, n, k, zero_points=zpk, nibble_format=K.NIBBLE_UNSIGNED)
    x = (torch.randn(m, k, generator=gen, device="cuda") * torch.logspace(-3, 3, m, device="cuda")[:, None]).to(dt)
    guard = torch.full((m * n + 64,), 7.0, device="cuda", dtype=dt)  # nothing is written behind the last row
    y = w.matmul(x, out=guard[:m * n].view(m, n))
    assert y.shape == (m, n) and y.dtype == dt and bool((guard[m * n:] == 7.0).all())
    q = torch.stack((b & 15, b >> 4), dim=2).reshape(n, k).float()
    zf = z[:, :groups].float().repeat_interleave(g, dim=1) if zp else 8.0
    wf = ((q - zf).half() * sc.repeat_interleave(g, dim=1)).double()
    xd = x.double()
    off = {"f32": 2.0 ** -23, "f16": 2.0 ** -11, "bf16": 2.0 ** -8}[act]
    rows = k * 2.0 ** -24 + (0.0 if act == "f16" else 2.0 ** -11)
    for c0 in range(0, n, 8192):
        want = xd @ wf[c0:c0 + 8192].t().contiguous()
        mag = xd.abs() @ wf[c0:c0 + 8192].abs().t().contiguous()
        err = (y[:, c0:c0 + 8192].double() - want).abs()
        tiny = xd.abs().amax(1, keepdim=True) * 1e-7
        assert bool((err <= mag * rows + want.abs() * off + tiny + 1e-7).all()), (c0, float((err / (mag + 1e-30)).max()))



@pytest.mark.parametrize("m,n,k", [(150, 28674, 192), (515, 14338, 320), (300, 4098, 4096)])
def test_epilogues(m, n, k):
    import torch

    from yscv_amd import kernels as K

    gen = torch.Generator(device="cuda").manual_seed(m)
    b = torch.randint(0, 256, (n * k // 2,), generator=gen, device="cuda", dtype=torch.uint8).cpu().numpy()
    sc = (torch.rand(n * (k // 32), generator=gen, device="cuda") * 0.015 + 0.005).half().cpu().numpy()
    w = K.PackedInt4Weight(b, sc, 32, n, k, nibble_format=K.NIBBLE_UNSIGNED)
    x = torch.randn(m, k, generator=gen, device="cuda").half()
    y = w.matmul(x, out_dtype=torch.float32)
    h = torch.randn(m, n, generator=gen, device="cuda")
    got = h.clone()
    w.matmul_fused(x, got, K.EPILOGUE_ADD_F32)
    assert bool(((got - (h + y)).abs() <= 1e-6 * (h.abs() + y.abs())).all())  # one f32 addition
    act = torch.empty(m, n // 2, device="cuda", dtype=torch.float16)
    w.matmul_fused(x, act, K.EPILOGUE_SWIGLU)
    gate, up = y[:, 0::2].double(), y[:, 1::2].double()
    want = gate * torch.sigmoid(gate) * up
    assert bool(((act.double() - want).abs() <= 2.0 ** -10 * want.abs() + 1e-6).all())  # fp16, and exp in f32
