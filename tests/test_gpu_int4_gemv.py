"""One activation row of each type, and up to four: every group form with and without zero points, waves that share a block of rows (one to
eight, and slices behind the eighth), K that ends inside a slice, rows that end inside a block or a group of blocks, and several
groups per workgroup.  Reference: the dequantised product in float64."""
import pytest

pytestmark = pytest.mark.gpu

CASES = [(n, k, g, scales, zp) for (n, k) in [(1, 256), (17, 768), (1000, 1280), (129, 2816), (50, 4864), (200, 13056)]
         for (g, scales, zp) in [(32, "f32", False), (64, "f16", True), (128, "f16", False), (256, "f32", True), (32, "f16", True)]]
CASES += [(33, 32, 32, "f16", False), (100, 96, 32, "f32", True), (77, 2880, 64, "f32", False),
          (70001, 96, 32, "f32", False), (33100, 2400, 32, "f16", True), (33100, 2112, 64, "f32", False),
          (65700, 2080, 32, "f16", False)]


def _problem(n, k, g, act, scales, zp, m=1):
    """the weight, its dense form and the activations"""
    import torch

    from yscv_amd import kernels as K

    gen = torch.Generator(device="cuda").manual_seed(n + k)
    q = torch.randint(0, 16, (n, k), generator=gen, device="cuda", dtype=torch.uint8)
    sc = (torch.rand(n, k // g, generator=gen, device="cuda") * 0.015 + 0.005).to({"f16": torch.float16, "f32": torch.float32}[scales])
    z = torch.full((n, k // g + (k // g) % 2), 8, device="cuda", dtype=torch.uint8)
    if zp:
        z[:, :k // g] = torch.randint(0, 16, (n, k // g), generator=gen, device="cuda", dtype=torch.uint8)
    w = K.PackedInt4Weight((q[:, 0::2] | (q[:, 1::2] << 4)).cpu().numpy(), sc.cpu().numpy(), g, n, k,
                           zero_points=(z[:, 0::2] | (z[:, 1::2] << 4)).cpu().numpy() if zp else None, nibble_format=K.NIBBLE_UNSIGNED)
    dense = (q.double() - z[:, :k // g].double().repeat_interleave(g, 1)) * sc.double().repeat_interleave(g, 1)
    x = torch.randn(m, k, generator=gen, device="cuda").to({"f16": torch.float16, "f32": torch.float32, "bf16": torch.bfloat16}[act])
    return w, dense, x


@pytest.mark.parametrize("act", ["f16", "f32", "bf16"])
@pytest.mark.parametrize("n,k,g,scales,zp", CASES)
def test_one_row(n, k, g, scales, zp, act):
    _check(n, k, g, scales, zp, act, 1)


# both sides of the rule, every group form, idle waves and several groups per workgroup
@pytest.mark.parametrize("act", ["f16", "f32", "bf16"])
@pytest.mark.parametrize("m,n,k,g,scales,zp", [
    (2, 33, 96, 32, "f32", True), (2, 1000, 1280, 64, "f16", False), (2, 50, 4864, 128, "f16", True), (2, 16400, 2112, 64, "f32", False),
    (2, 70001, 768, 32, "f16", False), (3, 1000, 2560, 32, "f16", True), (4, 129, 2816, 64, "f32", False), (4, 4096, 4096, 32, "f16", False),
    (3, 200, 13056, 128, "f16", False), (4, 50, 4864, 256, "f32", True), (4, 77, 2880, 64, "f16", True), (3, 100, 1024, 32, "f16", False)])
def test_two_to_four_rows(m, n, k, g, scales, zp, act):
    _check(n, k, g, scales, zp, act, m)


def _check(n, k, g, scales, zp, act, m):
    import torch

    w, dense, x = _problem(n, k, g, act, scales, zp, m)
    got = w.matmul(x, out_dtype=torch.float32)
    # products hold 22 bits of an f32 x (all of a 16-bit one) and the weight exactly; a zero point is subtracted behind the sum of
    # 32 products (up to 15 times their size); then come four additions and the rounding of the result: every rounding is at
    # most 2^-23 of a sum of magnitudes
    # (where the rule leaves the call to the skinny kernel, 16-bit rows with zero point 8 keep 1024 in the weights)
    slices, cus = -(-k // 512), torch.cuda.get_device_properties(0).multi_processor_count
    groups = -(-n // (16 * {1: 8, 2: 4, 3: 2, 4: 2}.get(slices, 1)))
    here = m == 1 or (slices <= 2 or groups <= 2 * cus if m == 2 else slices >= 5 and groups <= cus)
    bound = 2.0 ** -23 * ((32 if zp else 4) + 5 if here else 4096) * (x.double().abs() @ (dense.abs() + (dense.abs().mean() if zp else 0)).t())
    assert bool(((got.double() - x.double() @ dense.t()).abs() <= bound).all())
    for dt in (torch.float16, torch.bfloat16):
        assert torch.equal(w.matmul(x, out_dtype=dt), got.to(dt))


def test_magnitudes():
    """f32 rows far from one keep their relative accuracy, zeros give zeros."""
    import torch

    w, dense, x = _problem(300, 1536, 32, "f32", "f32", True)
    want = x.double() @ dense.t()
    for e in (-100, -30, 40):
        got = w.matmul(x * 2.0 ** e, out_dtype=torch.float32).double() * 2.0 ** -e
        assert float((got - want).norm() / want.norm()) < 2e-7  # about 1e-7 at one
    assert float(w.matmul(x * 0, out_dtype=torch.float32).abs().max()) == 0.0


@pytest.mark.parametrize("m,n,k", [(1, 40, 96), (1, 1002, 1056), (1, 520, 8736), (1, 33100, 2400), (2, 1002, 1056), (2, 40000, 768),
                                   (3, 1002, 2592), (4, 520, 8736)])
@pytest.mark.parametrize("act", ["f16", "f32"])
def test_epilogues(m, n, k, act):
    """residual update and SwiGLU against the plain product of the same kernel, and a workspace that is too small"""
    import torch

    from yscv_amd import kernels as K

    w, _, x = _problem(n, k, 32, act, "f16", False, m)
    v = w.matmul(x, out_dtype=torch.float32)
    h = torch.randn(m, n, device="cuda")
    y = h.clone()
    w.matmul_fused(x, y, K.EPILOGUE_ADD_F32)
    assert torch.equal(y, h + v)
    out = torch.empty(m, n // 2, device="cuda", dtype=torch.float16)
    w.matmul_fused(x, out, K.EPILOGUE_SWIGLU)
    ref = torch.nn.functional.silu(v[:, 0::2].double()) * v[:, 1::2].double()
    # one rounding to fp16 behind a silu whose exponential is good to a few units of 2^-22
    assert float(((out.double() - ref).abs() - (2.0 ** -11 + 2.0 ** -19) * ref.abs()).max()) <= 2.0 ** -24
    if k > 4096:  # (the kernel needs no workspace; the advertised size is for the others and still asked for)
        with pytest.raises(Exception, match="workspace"):
            w.matmul(x, out_dtype=torch.float32, workspace=torch.empty(256, dtype=torch.uint8, device="cuda"))
