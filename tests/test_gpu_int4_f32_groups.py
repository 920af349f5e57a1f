"""f32 activations against f32 scales above 16 rows: groups of 16 rows side by side give what the groups give one at a time."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k,g,zp,off", [(17, 358, 512, 64, False, 0), (33, 100, 96, 32, True, 0), (81, 358, 5056, 64, False, 0),
                                            (128, 4096, 4096, 32, False, 0), (127, 1000, 8192, 128, True, 0), (48, 300, 1024, 32, False, 1),
                                            (128, 70000, 4608, 64, False, 0), (20, 64, 2560, 128, True, 2)])
@pytest.mark.parametrize("out", ["f32", "f16"])
def test_groups_equal_separate_calls(m, n, k, g, zp, off, out):
    import torch

    from yscv_amd import kernels as K

    rng = np.random.default_rng(m + n + k)
    zpk = rng.integers(0, 256, n * ((k // g + 1) // 2), dtype=np.uint8) if zp else None
    w = K.PackedInt4Weight(rng.integers(0, 256, n * k // 2, dtype=np.uint8), rng.uniform(0.005, 0.02, n * (k // g)).astype(np.float32), g, n, k,
                           zero_points=zpk, nibble_format=K.NIBBLE_UNSIGNED)
    x = torch.empty(m * k + off, device="cuda")[off:].view(m, k)  # off: rows off 16-byte alignment
    x.copy_(torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)))
    odt = torch.float32 if out == "f32" else torch.float16
    y = w.matmul(x, out_dtype=odt)
    for r0 in range(0, m, 16):
        want = w.matmul(x[r0:r0 + 16], out_dtype=odt)
        if want.shape[0] > 4:
            assert torch.equal(y[r0:r0 + 16], want), r0
        else:  # up to four rows alone take another form: f32 sums of K products in another order, 2^-24 each
            d = (y[r0:r0 + 16].double() - want.double()).norm() / want.double().norm()
            assert float(d) <= (1e-5 if out == "f32" else 1e-3), r0
