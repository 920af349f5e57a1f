"""int8 GEMM in tiles of 64 x 128 and 128 x 256: whole numbers, so every value has to be the exact one.  K around the pairs of k-steps of 64,
the stages of four of them and the two or three stages in flight; rows and columns off the tiles; sums and bytes (the operators' forms of the
result: test_gpu_int8_forms.py)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# more 64 x 64 tiles than any CU count: rows x columns that take the small tile for few k-steps and the large one for many (sums from eight and two
# on, bytes from 24 and more on)
SMALL, LARGE = (1025, 4097), (2113, 8201)
KSTEPS = [2, 3, 4, 5, 6, 7, 8, 9, 11, 12, 13, 16, 17, 24]


def _case(torch, m, n, k, signed):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randint(-128, 128, (m, k), generator=g, device="cuda", dtype=torch.int8) if signed else \
        torch.randint(0, 256, (m, k), generator=g, device="cuda", dtype=torch.uint8)
    b = torch.randint(-128, 128, (k, n), generator=g, device="cuda", dtype=torch.int8)
    return a, b


@pytest.mark.parametrize("m,n", [SMALL, LARGE])
@pytest.mark.parametrize("ksteps", KSTEPS)
def test_sums_and_bytes(m, n, ksteps):
    import torch

    from yscv_amd import kernels as K

    signed, k = ksteps % 2 == 0 and ksteps > 8, 64 * ksteps - (1 if ksteps == 13 else 0)
    zp = -5 if signed else 129
    a, b = _case(torch, m, n, k, signed)
    w = K.pack_i8_b_for_matmul(b.cpu().numpy(), k, n)
    want = ((a.double() - zp) @ b.double()).to(torch.int32)  # below 2^53: exact
    assert torch.equal(w.matmul(a, a_zp=zp), want)
    comp = (torch.arange(n, device="cuda") % 7 + 4).float() * (8.0 / (74.0 * 73.0 * k ** 0.5))
    lo, hi = (-128, 127) if signed else (0, 255)
    for how in (K.ROUND_HALF_AWAY, K.ROUND_TIES_EVEN):
        v = want.float() * comp + 3.0
        t = torch.trunc(v)
        r = torch.where((v - t).abs() >= 0.5, t + torch.copysign(torch.ones_like(v), v), t) if how == K.ROUND_HALF_AWAY else torch.round(v)
        got = w.matmul_requant(a, zp, comp, 3.0, how, lo, hi)
        assert torch.equal(got.to(torch.int32), r.clamp(lo, hi).to(torch.int32))


@pytest.mark.parametrize("m,n", [(64, 128), SMALL, LARGE])
def test_requantised_infinities_and_nans(m, n):
    import torch

    from yscv_amd import kernels as K

    k = 192
    a, b = _case(torch, m, n, k, False)
    w = K.pack_i8_b_for_matmul(b.cpu().numpy(), k, n)
    want = ((a.double() - 128) @ b.double()).to(torch.int32)
    comp = torch.full((n,), 0.003, device="cuda")
    comp[0::5], comp[1::5], comp[2::5] = float("inf"), float("nan"), 3e38
    v = (want.float() * comp + 140.0).cpu().numpy()  # inf * 0 is a NaN too
    for lo, hi in ((0, 255), (128, 200), (3, 90)):
        with np.errstate(invalid="ignore"):
            t = np.trunc(v)
            r = np.where(np.abs(v - t) >= 0.5, t + np.copysign(np.float32(1.0), v), t)
            q = np.where(np.isnan(r), 0, np.minimum(np.maximum(r, lo), hi)).astype(np.int64)
        got = w.matmul_requant(a, 128, comp, 140.0, K.ROUND_HALF_AWAY, lo, hi).cpu().numpy()
        assert np.array_equal(got.astype(np.int64), q), (lo, hi)
