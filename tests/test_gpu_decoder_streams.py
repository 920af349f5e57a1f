"""Decoder calls on streams other than the default one: which are refused, and that calls follow each other whatever streams
they name."""
import numpy as np
import pytest

from test_gpu_decoder import PCFG

pytestmark = pytest.mark.gpu

MODES = {"launches": dict(use_graph=False), "graph": dict(use_graph=True), "single_launch": dict(persistent=True), "auto": dict(auto=True)}


def _decoder(**cfg):
    from yscv_amd.decoder import Decoder

    dec = Decoder(**dict(PCFG, **cfg))
    dec.init_random(seed=3, nibbles=(1, 15))
    return dec


@pytest.mark.parametrize("mode", [*MODES, "prefill"])
def test_a_captured_stream_is_refused_and_nothing_moves(mode):
    import torch

    from yscv_amd.capi import YscvHipError

    dec = _decoder()
    side = torch.cuda.Stream()

    def call(stream=None):
        if mode == "prefill":
            dec.prefill([5, 6, 7], stream=stream)
        else:
            dec.run(2, stream=stream, **MODES[mode])

    dec.reset([9], 0)
    call(side.cuda_stream)  # an earlier call on the same stream
    torch.cuda.synchronize()
    x = torch.zeros(4, device="cuda")
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        with pytest.raises(YscvHipError, match="captured"):
            call(side.cuda_stream)
        x += 1  # the capture itself goes on
    for _ in range(3):
        g.replay()
    torch.cuda.synchronize()
    assert x.tolist() == [3.0] * 4
    if mode != "prefill":  # the state is the one after the two steps
        want = _decoder()
        want.reset([9], 0)
        want.run(PCFG["max_steps"], **MODES[mode])
        dec.run(PCFG["max_steps"] - 2, **MODES[mode])
        assert np.array_equal(dec.tokens(0, PCFG["max_steps"]), want.tokens(0, PCFG["max_steps"]))
