"""int4 matmul of five to sixteen 16-bit rows: every number of 16-row blocks that a workgroup can end with, over its rounds of four with two
or four blocks in flight, rows that leave lanes without one, and a K whose last wave ends early or has nothing to do."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# blocks per workgroup 1 .. 8 (two in flight) and from 9 on (four), the last block cut
BLOCKS = [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 13]


@pytest.mark.parametrize("blocks", BLOCKS)
@pytest.mark.parametrize("m,k,dtype", [(16, 4096, "float16"), (5, 4096, "bfloat16"), (9, 1088, "float16"), (12, 8704, "bfloat16"), (8, 2080, "float16")])
def test_blocks_of_a_workgroup(blocks, m, k, dtype):
    import torch

    from yscv_amd import kernels as K

    cus = torch.cuda.get_device_properties(0).multi_processor_count
    slices = -(-k // 512)
    parts = -(-slices // 8)  # of K, over workgroups
    waves = -(-slices // parts)
    per = cus * max(1, 8 // (waves if waves <= 2 else 8)) // parts
    n, g = 16 * per * blocks - 5, 32
    gen = torch.Generator(device="cuda").manual_seed(blocks * 100 + m)
    packed = torch.randint(0, 256, (n, k // 2), generator=gen, device="cuda", dtype=torch.uint8)
    scales = (torch.rand(n, k // g, generator=gen, device="cuda") * 0.015 + 0.005).half()
    x = torch.randn(m, k, generator=gen, device="cuda").to(getattr(torch, dtype))
    w = K.PackedInt4Weight(packed.cpu().numpy().reshape(-1), scales.cpu().numpy().reshape(-1), g, n, k, nibble_format=K.NIBBLE_UNSIGNED)
    got = w.matmul(x, out_dtype=torch.float32).double()
    q = torch.stack([packed & 15, packed >> 4], dim=2).reshape(n, k)
    want = torch.empty(m, n, device="cuda", dtype=torch.float64)
    for r in range(0, n, 8192):  # in pieces: the weights in 64 bits are large
        s = slice(r, min(r + 8192, n))
        want[:, s] = x.double() @ ((q[s].double() - 8) * scales[s].double().repeat_interleave(g, dim=1)).t().contiguous()
    # products are exact; weights enter as 1024 + q or 64 + q, whose sums are taken back in f32: each of the roundings on a term's way is at
    # most 2^-24 of sum |x| (1024 + 15) scale, sixteen of them at worst (four MFMA steps, scale, four tiles, eight waves in a tree of three)
    bound = 16 * 2.0 ** -24 * 1039 * 0.02 * x.double().abs().sum(dim=1, keepdim=True)
    assert bool(((got - want).abs() <= bound).all()), float(((got - want).abs() / bound).max())
