"""int8 GEMM with a K of 64 and less, one step of the matrix cores, and more tiles than CUs: whole numbers, so every value has to be the
exact one, and a shorter K is not the slower call."""
import statistics

import pytest

pytestmark = pytest.mark.gpu

# more 64 x 64 tiles than a card has CUs: rows, columns or both of them many, off every tile, and one column block only
MANY = [(2113, 4097), (2113, 8201), (1025, 4097), (20000, 64), (20001, 1), (4097, 515), (65, 30000), (1, 70000)]


def _operands(torch, m, n, k, signed):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randint(-128, 128, (m, k), generator=g, device="cuda", dtype=torch.int8) if signed else \
        torch.randint(0, 256, (m, k), generator=g, device="cuda", dtype=torch.uint8)
    b = torch.randint(-128, 128, (k, n), generator=g, device="cuda", dtype=torch.int8)
    return a, b


@pytest.mark.parametrize("m,n", MANY)
@pytest.mark.parametrize("k,signed", [(64, False), (64, True), (63, False), (1, True)])
def test_sums_and_bytes(m, n, k, signed):
    import torch

    from yscv_amd import kernels as K

    a, b = _operands(torch, m, n, k, signed)
    zp, lo, hi = (-5, -128, 127) if signed else (129, 0, 255)
    w = K.pack_i8_b_for_matmul(b.cpu().numpy(), k, n)
    want = ((a.double() - zp) @ b.double()).to(torch.int32)  # below 2^53: exact
    assert torch.equal(w.matmul(a, a_zp=zp), want)
    comp = (torch.arange(n, device="cuda") % 7 + 4).float() * (8.0 / (74.0 * 73.0 * k ** 0.5))
    v = want.float() * comp + 3.0
    got = w.matmul_requant(a, zp, comp, 3.0, K.ROUND_TIES_EVEN, lo, hi)
    assert torch.equal(got.to(torch.int32), torch.round(v).clamp(lo, hi).to(torch.int32))


@pytest.mark.parametrize("m,n", [(20000, 64), (2048, 8192)])
def test_takes_no_longer_than_two_steps(m, n):
    import torch

    from yscv_amd import kernels as K

    us = {}
    for k in (64, 128):
        a, b = _operands(torch, m, n, k, False)
        w = K.pack_i8_b_for_matmul(b.cpu().numpy(), k, n)
        for _ in range(5):
            w.matmul(a, a_zp=128)
        spans = []
        for _ in range(9):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(10):
                w.matmul(a, a_zp=128)
            end.record()
            end.synchronize()
            spans.append(start.elapsed_time(end) * 100.0)
        us[k] = statistics.median(spans)
    # a kernel that walks such tiles by a round of the CUs for each 64 x 64 took 2.6 and 4.1 times as long
    assert us[64] <= 1.5 * us[128], us
