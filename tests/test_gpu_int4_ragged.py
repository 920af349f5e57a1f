"""int4 matmul at the edges of its kernels' tiles: K that ends inside a 512-k slice, a 128-k tile or a 64-k line, ragged
rows and columns, on the skinny kernel (m <= 16), the K-split kernel (its tile shapes and its split over workgroups), the
register-resident kernel for wide weights and the LDS-ring GEMM.  Reference: the dequantised product in float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _problem(m, n, k, g, act, scales, zp, seed):
    import torch

    from yscv_amd import kernels as K

    gen = torch.Generator(device="cuda").manual_seed(seed)
    q = torch.randint(0, 16, (n, k), generator=gen, device="cuda", dtype=torch.uint8)
    sc = (torch.rand(n, k // g, generator=gen, device="cuda") * 0.015 + 0.005).to({"f16": torch.float16, "f32": torch.float32}[scales])
    z = torch.randint(5, 12, (n, k // g), generator=gen, device="cuda", dtype=torch.uint8) if zp else None
    packed_z = None
    if zp:
        zz = torch.cat([z, torch.full((n, (k // g) % 2), 8, device="cuda", dtype=torch.uint8)], 1)
        packed_z = (zz[:, 0::2] | (zz[:, 1::2] << 4)).cpu().numpy()
    w = K.PackedInt4Weight((q[:, 0::2] | (q[:, 1::2] << 4)).cpu().numpy(), sc.cpu().numpy(), g, n, k, zero_points=packed_z,
                           nibble_format=K.NIBBLE_UNSIGNED)
    dense = (q.double() - (z.double() if zp else torch.full((n, k // g), 8.0, device="cuda", dtype=torch.float64)).repeat_interleave(g, 1)) * \
        sc.double().repeat_interleave(g, 1)
    x = torch.randn(m, k, generator=gen, device="cuda").to({"f16": torch.float16, "f32": torch.float32, "bf16": torch.bfloat16}[act])
    return w, x, x.double() @ dense.t()


CASES = [
    # m, n, k, group, activations, scales, zero points
    (1, 33, 32, 32, "f16", "f16", False), (1, 1000, 1376, 32, "f32", "f32", False), (4, 257, 2912, 32, "f32", "f16", True),
    (3, 4096, 544, 32, "bf16", "f16", False), (7, 100, 4192, 32, "f16", "f16", False), (16, 333, 960, 64, "bf16", "f16", True),
    (16, 200, 4736, 128, "f32", "f32", False), (9, 64, 1056, 32, "f32", "f16", False),
    # one pair of k-steps, half a pair, fewer tiles than waves
    (17, 16, 32, 32, "f16", "f16", False), (33, 50, 64, 64, "f16", "f16", True), (40, 100, 96, 32, "bf16", "f16", False),
    (64, 128, 1024, 128, "f16", "f16", True),
    # each tile shape, ragged in every direction
    (31, 1001, 1056, 32, "f16", "f16", False), (32, 4099, 2880, 64, "f16", "f16", True), (20, 14300, 4096, 32, "f16", "f16", False),
    (65, 1003, 1312, 32, "f16", "f16", False), (100, 3001, 2880, 64, "bf16", "f16", False), (200, 3001, 4160, 64, "f16", "f16", True),
    (250, 1111, 4128, 32, "f32", "f16", False), (120, 130, 8320, 128, "f16", "f16", False), (77, 515, 1056, 32, "f16", "f32", False),
    # K also split over workgroups
    (24, 1000, 14336, 32, "f16", "f16", False), (64, 520, 14368, 32, "f16", "f16", True), (130, 1030, 11008, 128, "bf16", "f16", False),
    # more column blocks than CUs: the register-resident kernel and the LDS-ring GEMM, K not a multiple of 64 among them
    (18, 30001, 1056, 32, "f16", "f16", False), (32, 20000, 4640, 32, "bf16", "f16", True), (150, 14336, 1120, 32, "f16", "f16", False),
    (300, 6001, 992, 32, "bf16", "f16", True),
]


@pytest.mark.parametrize("m,n,k,g,act,scales,zp", CASES)
def test_product(m, n, k, g, act, scales, zp):
    import torch

    w, x, want = _problem(m, n, k, g, act, scales, zp, m * 31 + n + k)
    got = w.matmul(x, out_dtype=torch.float32)
    rel = float((got.double() - want).norm() / want.norm())
    exact = act == "f32" and (scales == "f32" or m <= 16)
    assert rel < (1e-5 if exact else 6e-4), rel
    assert float((got.double() - want).abs().max()) < (2e-5 if exact else 6e-3) * float(want.abs().max())
    assert torch.equal(got, w.matmul(x, out_dtype=torch.float32))
    # rows must not see what lies behind them: the same rows with a NaN row after the last one
    buf = torch.full((m + 1, k), float("nan"), device="cuda", dtype=x.dtype)
    buf[:m] = x
    assert torch.equal(w.matmul(buf[:m], out_dtype=torch.float32), got)
    # activations on an odd alignment, with a workspace of the advertised size where K needs padding then
    ws = torch.empty(max(w.workspace_bytes(m, x.dtype), 256), dtype=torch.uint8, device="cuda")
    odd = torch.empty(m * k + 1, device="cuda", dtype=x.dtype)
    odd[1:] = x.reshape(-1)
    shifted = w.matmul(odd[1:].view(m, k), out_dtype=torch.float32, workspace=ws if k % 512 else None)
    assert float((shifted.double() - want).norm() / want.norm()) < (1e-5 if exact else 6e-4)


@pytest.mark.parametrize("m,n,k", [(40, 1002, 1056), (64, 520, 14368), (100, 3002, 2880), (18, 30002, 1056)])
def test_epilogues(m, n, k):
    import torch

    from yscv_amd import kernels as K

    w, x, want = _problem(m, n, k, 32, "f16", "f16", False, 5)
    h = torch.randn(m, n, device="cuda")
    y = h.clone()
    w.matmul_fused(x, y, K.EPILOGUE_ADD_F32)
    assert float((y.double() - h.double() - want).norm() / want.norm()) < 6e-4
    act = torch.empty(m, n // 2, device="cuda", dtype=torch.float16)
    w.matmul_fused(x, act, K.EPILOGUE_SWIGLU)
    ref = torch.nn.functional.silu(want[:, 0::2]) * want[:, 1::2]
    assert float((act.double() - ref).norm() / ref.norm()) < 2e-3
