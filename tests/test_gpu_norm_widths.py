"""RMSNorm on both sides of the widths up to which a row waits in the registers of its workgroup: the entry point on f32 tensors, rows that
end inside a load of 256 threads, rows that start off sixteen bytes, and values past the ends of a row that must not count."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [4, 12, 1020, 1024, 1028, 4092, 4096, 4100, 8188, 8192, 8196, 1023, 4097])
@pytest.mark.parametrize("offset", [0, 1])
def test_against_64_bits(d, offset):
    import torch

    from yscv_amd import onnx_ops as O

    rng = np.random.default_rng(d)
    rows = 5
    x = rng.standard_normal((rows, d)).astype(np.float32)
    x[1] *= 1e-3
    x[2, -1] = np.inf  # stays in its own row
    x[4, 0] = np.nan
    gamma = rng.uniform(0.5, 1.5, d).astype(np.float32)
    buf = torch.zeros(rows * d + 8, device="cuda")
    xt = buf[offset:offset + rows * d].view(rows, d)
    xt.copy_(torch.from_numpy(x))
    y = O.rms_norm(xt, torch.from_numpy(gamma).cuda(), 1e-5).cpu().numpy()
    for r in (0, 1, 3):
        x64 = x[r].astype(np.float64)
        want = x64 / np.sqrt((x64 * x64).mean() + 1e-5) * gamma
        # half an ulp each for two products, quotient, root and quotient; the sum of squares (all positive) has at most 32 additions of a
        # thread and eight of the reduction on one path, and the root halves its error.  Longer rows than 8192 values: no more per thread.
        assert np.abs(y[r] - want).max() <= (5 + 40 / 2) * 2.0**-24 * np.abs(want).max() * 1.01
    assert np.isnan(y[2, -1]) and np.all(y[2, :-1] == 0)
    assert np.isnan(y[4]).all()
