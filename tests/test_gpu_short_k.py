"""Weights of K up to 1024: several skinny workgroups to a CU, and decode steps of such widths whose folded norms cover up to sixteen rows
with one or two waves."""
import numpy as np
import pytest

from test_gpu_decoder import LOGIT_TOL, _build
from test_gpu_decoder_fold import BASE, SHAPES

pytestmark = pytest.mark.gpu


# (m, n, k, group, act, scales, zero points): fewer blocks than workgroups, one each, several with a remainder, groups of 16 rows
@pytest.mark.parametrize("m,n,k,g,act,sdt,zp", [
    (16, 300, 512, 32, "f16", "f16", False), (9, 4113, 1024, 32, "f16", "f16", True), (16, 16400, 1024, 64, "bf16", "f16", False),
    (5, 33001, 96, 32, "f16", "f16", False), (13, 40017, 896, 128, "f16", "f16", False), (14, 20003, 576, 64, "f32", "f32", False),
    (6, 50000, 1024, 32, "f32", "f16", True), (2, 30001, 512, 32, "bf16", "f16", False), (40, 20001, 512, 32, "f32", "f32", False),
    (130, 9000, 1024, 128, "f32", "f32", True)])
def test_matmul_against_64_bits(m, n, k, g, act, sdt, zp):
    import torch

    from yscv_amd import kernels as K

    dt = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    groups = k // g
    b = torch.randint(0, 256, (n, k // 2), generator=gen, device="cuda", dtype=torch.uint8)
    sc = (torch.rand(n, groups, generator=gen, device="cuda") * 0.015 + 0.005).to(dt[sdt])
    z = torch.randint(0, 16, (n, (groups + 1) // 2 * 2), generator=gen, device="cuda", dtype=torch.uint8) if zp else None
    zpk = (z[:, 0::2] | (z[:, 1::2] << 4)).reshape(-1).cpu().numpy() if zp else None
    w = K.PackedInt4Weight(b.reshape(-1).cpu().numpy(), sc.reshape(-1).cpu().numpy(), g, n, k, zero_points=zpk, nibble_format=K.NIBBLE_UNSIGNED)
    x = torch.randn(m, k, generator=gen, device="cuda").to(dt[act])
    y = w.matmul(x, out_dtype=torch.float32).double()
    q = torch.stack((b & 15, b >> 4), dim=2).reshape(n, k).double()
    zf = z[:, :groups].double().repeat_interleave(g, dim=1) if zp else 8.0
    wf = (q - zf) * sc.double().repeat_interleave(g, dim=1)
    xa = x.double().abs()
    want, mag = x.double() @ wf.t().contiguous(), xa @ wf.abs().t().contiguous()
    # f32 sums.  fp16 rows meet 1024 + q or 64 + q, and the offset goes from the sums of 32: each is off by up to 34 roundings of 2^-24 of
    # 1040 |x|, in front of its scale.  f32 rows go as fp16 hi + lo, 2^-22 of a value.
    off = xa @ (sc.double().repeat_interleave(g, dim=1) * 1040.0).t().contiguous()
    assert bool(((y - want).abs() <= mag * (k * 2.0 ** -24 + 2.0 ** -21) + off * (0.0 if act == "f32" or zp else 34 * 2.0 ** -24) + 1e-6).all())


@pytest.mark.parametrize("name,batch", [("k2816", 9), ("k2816", 16), ("k768", 16), ("one_slice", 13)])
def test_steps_match_numpy(name, batch):
    rng = np.random.default_rng(8100 + batch)
    cfg = dict(BASE, **SHAPES[name], max_batch=batch)
    dec, ref = _build(rng, cfg, symmetric=True)
    tok = rng.integers(0, cfg["vocab"], batch).astype(np.int32)
    dec.reset(tok, 0)
    for step in range(4):
        dec.run(1, use_graph=bool(step & 1))
        exp, got = ref.step(tok, step), dec.logits()
        assert float(np.abs(got - exp).max() / np.abs(exp).max()) < LOGIT_TOL, step
        tok = dec.tokens(step, 1)[0].copy()
