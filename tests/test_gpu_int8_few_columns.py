"""int8 GEMM of many rows and few columns, fewer column blocks than the chip has dies: whole numbers, so every value has to be the exact one, and no
slower than the same product the other way round."""
import statistics

import pytest

pytestmark = pytest.mark.gpu


def _operands(torch, m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randint(0, 256, (m, k), generator=g, device="cuda", dtype=torch.uint8)
    return a, torch.randint(-128, 128, (k, n), generator=g, device="cuda", dtype=torch.int8)


@pytest.mark.parametrize("m,n,k", [(3419, 16, 7616), (1912, 160, 1664), (4299, 50, 1858), (2450, 112, 1280), (1089, 80, 7488), (2314, 128, 192), (129, 700, 640),
                                   (1, 16, 64), (17, 129, 64), (255, 1040, 2112)])
def test_every_value(m, n, k):
    import torch

    from yscv_amd import kernels as K

    a, b = _operands(torch, m, n, k)
    w = K.pack_i8_b_for_matmul(b.cpu().numpy(), k, n)
    assert torch.equal(w.matmul(a, a_zp=131), ((a.double() - 131) @ b.double()).to(torch.int32))


@pytest.mark.parametrize("m,n,k", [(3419, 16, 7616), (1912, 160, 1664)])
def test_takes_no_longer_than_few_rows_and_many_columns(m, n, k):
    import torch

    from yscv_amd import kernels as K

    us = []
    for rows, cols in ((m, n), (n, m)):
        a, b = _operands(torch, rows, cols, k)
        w = K.pack_i8_b_for_matmul(b.cpu().numpy(), k, cols)
        for _ in range(5):
            w.matmul(a, a_zp=128)
        spans = []
        for _ in range(9):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(20):
                w.matmul(a, a_zp=128)
            end.record()
            end.synchronize()
            spans.append(start.elapsed_time(end) * 50.0)
        us.append(statistics.median(spans))
    # with whole column blocks on each die it was 6 and 1.8 times as long
    assert us[0] <= 1.5 * us[1], us
