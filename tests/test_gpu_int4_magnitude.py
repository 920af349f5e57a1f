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


def test_single_launch_decoder_with_small_activations():
    """The LM head of the single-launch decode path behind a norm whose gain leaves values of about 1e-5: against the
    multi-kernel path with its norms as launches of their own, which rounds the same fp16 (the folded norm rounds a quarter
    of it, whose last bit is four times as coarse).  That last bit is 2^-24: rounding is 2^-24 / sqrt(12) of 1e-5, 1.7e-3 of
    the result, on each side, and the paths' other rounding points add about 1e-3."""
    from test_gpu_decoder import PCFG
    from yscv_amd import lib
    from yscv_amd.decoder import Decoder

    dec = Decoder(**PCFG)
    dec.init_random(seed=3, nibbles=(1, 15))
    dec.set_norm(0, "final", np.full(PCFG["d_model"], 1e-5, np.float32))
    dec.finalize()
    lib().decoder_debug_set_folded_norm(dec._h, 0)
    logits = {}
    for name, kw in {"graph": dict(use_graph=True), "single": dict(persistent=True)}.items():
        dec.reset([9], 0)
        dec.run(1, **kw)
        logits[name] = dec.logits()[0].astype(np.float64)
    rel = np.linalg.norm(logits["single"] - logits["graph"]) / np.linalg.norm(logits["graph"])
    assert rel < 5e-3, rel
