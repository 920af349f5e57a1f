"""int4 matmul of fp16 rows of any magnitude: attention and SwiGLU outputs have many values below 2^-10, and the product has
to be that of the values as they are, down to fp16's own subnormals.  Reference: the dequantised product in float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,g", [(520, 2880, 64), (515, 2816, 32), (300, 4096, 32), (130, 11008, 128)])
@pytest.mark.parametrize("std", [1e4, 1.0, 1e-3, 1e-4, 1e-5])
def test_fp16_rows_of_any_magnitude(n, k, g, std):
    import torch

    from yscv_amd import kernels as K

    rng = np.random.default_rng(n + k)
    q = rng.integers(0, 16, (n, k), dtype=np.uint8)
    sc = rng.uniform(0.005, 0.02, (n, k // g)).astype(np.float16)
    w = K.PackedInt4Weight((q[:, 0::2] | (q[:, 1::2] << 4)).reshape(-1), sc.reshape(-1), g, n, k, nibble_format=K.NIBBLE_UNSIGNED)
    dense = (q.astype(np.float64) - 8.0) * sc.astype(np.float64).repeat(g, 1)
    x = np.clip(rng.standard_normal((40, k)) * std, -65504, 65504).astype(np.float16)
    want = x.astype(np.float64) @ dense.T
    xd = torch.from_numpy(x).cuda()
    for m in (1, 4, 5, 8, 9, 16, 17, 40):
        got = w.matmul(xd[:m], out_dtype=torch.float32).cpu().numpy().astype(np.float64)
        rel = np.linalg.norm(got - want[:m]) / np.linalg.norm(want[:m])
        # up to 16 rows the scales are applied in f32; what is left is the f32 rounding of a group's sum, whose terms
        # x (1024 + q) are up to 160 times the group's product, over a few roundings: 160 * 2^-24 * 5.  Above, the
        # weights are rounded to fp16.
        assert rel < (5e-5 if m <= 16 else 6e-4), (m, rel)
