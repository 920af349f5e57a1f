"""All layers of a small decoder's step in one launch (decode_layers.hip, what run(auto=True) takes at batch 1 where the shape
fits) against the numpy restatement and against the multi-kernel path."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_decoder import LOGIT_TOL, _build

pytestmark = pytest.mark.gpu

BASE = dict(n_layers=2, vocab=320, group_size=32, head_dim=64, max_batch=1, max_ctx=384, max_steps=16, rope_theta=10000.0, rms_eps=1e-5)
SHAPES = {
    "widest": dict(d_model=1024, n_heads=16, n_kv_heads=2, d_ff=2816),                # 2 / 1 / 6 / 3 tiles per wave, not all used
    "all_tiles": dict(d_model=1024, n_heads=16, n_kv_heads=8, d_ff=3072),             # every tile of every wave used
    "least": dict(d_model=128, n_heads=2, n_kv_heads=1, d_ff=128),                    # one wave with a tile, eight workgroups
    "sixteen_heads_per_kv_head": dict(d_model=640, n_heads=16, n_kv_heads=1, d_ff=1920),
    "one_head_per_kv_head": dict(d_model=384, n_heads=4, n_kv_heads=4, d_ff=640, rope_theta=500.0),
}


def _filled(name, start, seed, **over):
    rng = np.random.default_rng(seed)
    cfg = dict(BASE, **SHAPES[name], **over)
    dec, ref = _build(rng, cfg, symmetric=True, qkv_bias=name == "all_tiles")
    for l in range(cfg["n_layers"]):
        if start:
            k = rng.standard_normal((1, start, cfg["n_kv_heads"], 64)).astype(np.float16)
            v = rng.standard_normal((1, start, cfg["n_kv_heads"], 64)).astype(np.float16)
            dec.set_kv(l, k, v)
            ref.set_kv(l, k.astype(np.float32), v.astype(np.float32))
    return cfg, dec, ref


# positions at both ends of a wave's 32, a work item's 256 and a slab's 8; 2303 is nine work items for eight workgroups
@pytest.mark.parametrize("name,start", [("widest", 0), ("widest", 30), ("widest", 255), ("all_tiles", 6), ("all_tiles", 1022), ("least", 0),
                                        ("least", 62), ("least", 2303), ("sixteen_heads_per_kv_head", 254), ("one_head_per_kv_head", 29),
                                        ("one_head_per_kv_head", 380)])
def test_steps_match_numpy_and_the_multi_kernel_path(name, start):
    cfg, dec, ref = _filled(name, start, 6000 + start, max_ctx=(start + 4 + 127) // 128 * 128)
    tok = np.array([7], np.int32)
    dec.reset(tok, start)
    for step in range(3):
        dec.run(1, auto=True)
        exp = ref.step(tok, start + step)
        got = dec.logits()
        assert np.abs(got - exp).max() / np.abs(exp).max() < LOGIT_TOL, step
        assert dec.tokens(step, 1)[0, 0] == np.flatnonzero(got[0] == got.max())[-1]
        acts = {w: dec.activation(w).copy() for w in ("residual", "normed", "qkv", "attn_out", "ffn")}
        tok = dec.tokens(step, 1)[0].copy()
    for l in range(cfg["n_layers"]):
        gk, gv = dec.get_kv(l, 1, 0, start + 3)
        ek, ev = ref.kc[l][0][: start + 3], ref.vc[l][0][: start + 3]
        assert np.abs(gk.astype(np.float32) - ek).max() <= 1e-2 * np.abs(ek).max(), l
        assert np.abs(gv.astype(np.float32) - ev).max() <= 1e-2 * np.abs(ev).max(), l
    # the last step again as separate kernels: the same cache rows, the same activations to a few fp16 roundings per layer
    last_in = np.array([7], np.int32) if dec.tokens(0, 3).shape[0] < 2 else dec.tokens(1, 1)[0].copy()
    dec.reset(last_in, start + 2)
    dec.run(1, use_graph=False)
    one = dec.logits()
    assert np.abs(got - one).max() / np.abs(one).max() < 2e-3
    for which, a in acts.items():
        b = dec.activation(which)
        assert np.abs(a - b).max() <= 4e-3 * np.abs(b).max(), which


def test_the_same_bits_every_time_on_any_stream_and_across_the_end_of_the_tags():
    import torch

    from yscv_amd.capi import lib

    cfg, dec, _ = _filled("widest", 40, 6100, max_steps=64)
    n = 24

    def drive(stream=None, parts=(n,)):
        dec.reset(np.array([7], np.int32), 40)
        for p in parts:
            dec.run(p, auto=True, stream=stream)
        return dec.tokens(0, n).copy(), dec.logits().copy()

    want = drive()
    side = torch.cuda.Stream()
    last = 0xFFFFFFFE // (cfg["n_layers"] + 1) - 1  # the count of steps at which the entries are cleared
    for k, (stream, parts) in enumerate([(None, (1,) * n), (side.cuda_stream, (5, 19)), (None, (n,)), (None, (10, 14))]):
        if k >= 2:
            assert lib().decoder_debug_set_tag_epoch(dec._h, C.c_uint32(last - 12)) in (None, 0)
        tok, log = drive(stream, parts)
        assert np.array_equal(tok, want[0]) and np.array_equal(log, want[1]), k
    # another batch in between uses and replaces the other captured step only
    dec.reset(np.array([7], np.int32), 40)
    dec.run(2, use_graph=True)
    assert np.array_equal(drive()[1], want[1])
