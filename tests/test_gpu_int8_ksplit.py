"""int8 GEMM on shapes with few tiles (the K-split kernel) and on rows that are no multiple of 64 bytes (copied first):
whole numbers, so every value has to be the exact one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (m, k, n): each tile shape (1 .. 4 row tiles x 1 .. 4 column blocks) with one row or column more or less than a tile, k-steps
# fewer than waves, odd k-step counts, one pair per wave and many, and K around 64 and 128
SHAPES = [
    (1, 64, 16), (1, 1, 1), (1, 63, 17), (2, 65, 15), (15, 127, 33), (16, 128, 4096), (17, 129, 300), (1, 8192, 257), (16, 4160, 4097),
    (33, 192, 2050), (31, 1088, 4111), (32, 1023, 8190), (63, 4096, 4096), (65, 1000, 2000), (64, 8191, 65), (127, 320, 4095),
    (129, 1024, 4100), (197, 768, 3072), (197, 3072, 768), (256, 704, 4096), (511, 1216, 301), (1025, 768, 770), (2048, 257, 510),
    (4097, 64, 33), (600, 321, 4099), (1500, 4097, 1900),  # the last two: larger tiles on copied rows
]


def _inputs(torch, rng, m, k, n, signed):
    a = rng.integers(-128, 128, (m, k)).astype(np.int8) if signed else rng.integers(0, 256, (m, k)).astype(np.uint8)
    b = rng.integers(-128, 128, (k, n)).astype(np.int8)
    return a, b


def _exact(a, b, zp):
    return (a.astype(np.float64) - zp) @ b.astype(np.float64)  # below 2^53: exact


@pytest.mark.parametrize("m,k,n", SHAPES)
@pytest.mark.parametrize("signed", [False, True])
def test_sums_and_requantised_bytes(m, k, n, signed):
    import torch

    from yscv_amd import kernels as K

    rng = np.random.default_rng(m * 131 + k * 7 + n + signed)
    a, b = _inputs(torch, rng, m, k, n, signed)
    zp = -3 if signed else 131
    w = K.pack_i8_b_for_matmul(b, k, n)
    at = torch.from_numpy(a).cuda()
    want = _exact(a, b, zp)
    got = w.matmul(at, a_zp=zp)
    assert np.array_equal(got.cpu().numpy(), want.astype(np.int32))
    comp = (rng.uniform(0.5, 1.5, n) * 40.0 / (74.0 * 73.0 * np.sqrt(k))).astype(np.float32)
    corr = rng.integers(-500, 500, n).astype(np.int32)
    v = (want.astype(np.int64) + corr).astype(np.float32) * comp + np.float32(3.0)
    lo, hi = (-128, 127) if signed else (0, 255)
    q = np.clip(np.trunc(v) + np.where(np.abs(v - np.trunc(v)) >= 0.5, np.copysign(1.0, v), 0.0), lo, hi)
    got = w.matmul_requant(at, zp, torch.from_numpy(comp).cuda(), 3.0, K.ROUND_HALF_AWAY, lo, hi, corr=torch.from_numpy(corr).cuda())
    assert np.array_equal(got.cpu().numpy().astype(np.int64), q.astype(np.int64))


@pytest.mark.parametrize("m,k,n", [(5, 128, 64), (100, 1024, 520), (40, 77, 130)])
@pytest.mark.parametrize("off_a,off_out", [(1, 0), (8, 0), (0, 4), (3, 12)])
def test_tensors_off_16_byte_alignment(m, k, n, off_a, off_out):
    import torch

    from yscv_amd import kernels as K

    rng = np.random.default_rng(m + k + n + off_a)
    a, b = _inputs(torch, rng, m, k, n, False)
    w = K.pack_i8_b_for_matmul(b, k, n)
    buf = torch.empty(m * k + off_a, dtype=torch.uint8, device="cuda")
    at = buf[off_a:].view(m, k)
    at.copy_(torch.from_numpy(a))
    guard = torch.full((m * n + off_out // 4 + 4,), -77, dtype=torch.int32, device="cuda")
    out = guard[off_out // 4:off_out // 4 + m * n].view(m, n)
    w.matmul(at, a_zp=9, out=out)
    assert np.array_equal(out.cpu().numpy(), _exact(a, b, 9).astype(np.int32))
    assert (guard[:off_out // 4] == -77).all() and (guard[off_out // 4 + m * n:] == -77).all()


@pytest.mark.parametrize("m,k,n", [(7, 100, 48), (130, 333, 70), (300, 65, 2100)])
def test_f32_operators_with_copied_rows(m, k, n):
    """The operators that hold a scratch block while the GEMM copies its rows."""
    import torch

    from yscv_amd import onnx_ops as O

    rng = np.random.default_rng(m + k)
    b = rng.integers(-127, 128, (k, n)).astype(np.float32)
    x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).cuda()
    w = O.PrepackedI8B(torch.from_numpy(b).cuda())
    got, scale, zp = O.exec_dql_matmul_integer(x, w)
    q, s2, z2 = O.exec_dynamic_quantize_linear(x)
    assert float(scale) == float(s2) and float(zp) == float(z2)
    want = (q.cpu().numpy().astype(np.float64).reshape(m, k) - float(zp)) @ b.astype(np.float64)
    assert np.array_equal(got.cpu().numpy().reshape(m, n), want.astype(np.float32))


def test_a_long_matrix_is_copied_in_bounded_pieces():
    """800 MB of rows with a K that is no multiple of 64: the copy stays within the 64 MB block that is kept."""
    import torch

    from yscv_amd import kernels as K

    rng = np.random.default_rng(3)
    m, k, n = 200_003, 4001, 48
    b = rng.integers(-127, 128, (k, n), dtype=np.int8)
    w = K.pack_i8_b_for_matmul(b, k, n)
    a = torch.randint(0, 256, (m, k), device="cuda", dtype=torch.uint8)
    out = torch.empty(m, n, device="cuda", dtype=torch.int32)
    free = torch.cuda.mem_get_info()[0]
    w.matmul(a, a_zp=7, out=out)
    torch.cuda.synchronize()
    assert free - torch.cuda.mem_get_info()[0] <= 160 << 20  # the block and what the allocator rounds up to
    step = (64 << 20) // 4032 // 16 * 16
    rows = [0, m - 1] + [r for at in range(step, m, step) for r in (at - 1, at)]
    want = _exact(a[rows].cpu().numpy(), b, 7)
    assert np.array_equal(out[rows].cpu().numpy(), want.astype(np.int32))


@pytest.mark.parametrize("m,k,n", [(40, 77, 130), (300, 1001, 520)])
def test_capture_of_rows_that_would_be_copied(m, k, n):
    """A graph needs no memory for them: the kernel that reads any row runs there, with the same bytes as a result."""
    import torch

    from yscv_amd import kernels as K

    rng = np.random.default_rng(m)
    a, b = _inputs(torch, rng, m, k, n, False)
    w = K.pack_i8_b_for_matmul(b, k, n)
    at = torch.from_numpy(a).cuda()
    out = torch.zeros(m, n, dtype=torch.int32, device="cuda")
    w.matmul(at, a_zp=9, out=out)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        w.matmul(at, a_zp=9, out=out)
    for turn in range(3):
        new = torch.from_numpy(rng.integers(0, 256, (m, k), dtype=np.uint8))
        at.copy_(new)
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), _exact(new.numpy(), b, 9).astype(np.int32)), turn
