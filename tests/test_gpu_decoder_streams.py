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


def _hip():
    """The runtime this process already has loaded."""
    import ctypes as C

    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    hip = C.CDLL(path)
    hip.hipStreamCreateWithFlags.argtypes = [C.POINTER(C.c_void_p), C.c_uint]
    hip.hipStreamDestroy.argtypes = [C.c_void_p]
    return hip, C


@pytest.mark.parametrize("mode", MODES)
def test_calls_on_changing_streams_follow_each_other(mode):
    """reset, run, run_projections and prefill on the default stream, on streams that do not wait for it, and on streams that
    are destroyed right behind the call (their handles come back for the next ones), with no wait in between."""
    import torch

    dec = _decoder()
    prompt = np.arange(60, dtype=np.int32) * 7 % PCFG["vocab"]
    kw = MODES[mode]

    def drive(streams):
        dec.reset([9], 0)
        for s in streams[:5]:
            dec.run(3, stream=s(), **kw)
        first = dec.tokens(0, 15).copy(), dec.logits().copy()
        dec.prefill(prompt, stream=streams[5]())
        dec.run(4, stream=streams[6](), **kw)
        dec.reset([11], 64)
        dec.run(6, stream=streams[7](), **kw)
        last = dec.tokens(0, 6).copy(), dec.logits().copy()
        dec.prefill(prompt, stream=streams[8]())
        dec.run_projections(1, stream=streams[9]())  # leaves the cache and the tokens alone
        dec.run(5, stream=streams[10](), **kw)
        return first, last, (dec.tokens(0, 6).copy(), dec.logits().copy())

    want = drive([lambda: None] * 11)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    hip, C = _hip()
    alive = []

    def fresh():  # the stream before this one is destroyed now, right behind the call that used it
        while alive:
            assert hip.hipStreamDestroy(alive.pop()) == 0
        h = C.c_void_p()
        assert hip.hipStreamCreateWithFlags(C.byref(h), 1) == 0  # hipStreamNonBlocking
        alive.append(h)
        return h.value

    on_a, on_b, default = (lambda: a.cuda_stream), (lambda: b.cuda_stream), (lambda: None)
    for streams in ([on_a, on_b, on_a, on_a, default, on_b, on_a, on_b, default, on_a, on_b], [fresh] * 11,
                    [default, fresh, fresh, default, on_a, fresh, default, fresh, on_b, default, fresh]):
        for (tok, log), (wtok, wlog) in zip(drive(streams), want):
            assert np.array_equal(tok, wtok) and np.array_equal(log, wlog)
    torch.cuda.synchronize()
    while alive:
        assert hip.hipStreamDestroy(alive.pop()) == 0


def test_a_step_is_captured_again_behind_replays_under_way():
    """Changing the batch drops the captured step; its replays run to their end first."""
    import torch

    a, b = _decoder(), _decoder()
    side = torch.cuda.Stream()
    for turn in range(4):
        for tokens in ([9 + turn], [9 + turn, 40 + turn]):
            a.reset(tokens, 0)
            a.run(20, stream=side.cuda_stream)  # graph replays; the next turn's capture comes right behind them
        b.reset([9 + turn, 40 + turn], 0)
        b.run(20, use_graph=False)
        assert np.array_equal(a.tokens(0, 20), b.tokens(0, 20)) and np.array_equal(a.logits(), b.logits())


def test_a_failed_call_leaves_the_state_as_it_was():
    import torch

    from yscv_amd.capi import YscvHipError

    side = torch.cuda.Stream()
    dec = _decoder()
    dec.reset([9], 500)
    dec.run(12, auto=True)
    want = dec.tokens(0, 12).copy()
    for kw in MODES.values():
        dec.reset([9], 500)
        dec.run(5, stream=side.cuda_stream, **kw)
        for bad in (lambda: dec.run(8, stream=side.cuda_stream, **kw),           # past the end of the context
                    lambda: dec.run(1000, **kw),
                    lambda: dec.run(-1, **kw),
                    lambda: dec.prefill([1, PCFG["vocab"]], stream=side.cuda_stream),  # no such token
                    lambda: dec.prefill([1] * 20, start_pos=500),
                    lambda: dec.reset([1], PCFG["max_ctx"]),
                    lambda: dec.reset([1, 2, 3], 0)):
            with pytest.raises(YscvHipError):
                bad()
        dec.batch = 1
        dec.run(7, stream=side.cuda_stream, **kw)
        if "persistent" in kw or "auto" in kw:
            assert np.array_equal(dec.tokens(0, 12), want)
        else:
            assert dec.tokens(0, 12).shape == (12, 1)
        with pytest.raises(YscvHipError):
            dec.run(1, **kw)  # position 512 of 512


@pytest.mark.parametrize("n", [895, 896, 897, 1793])
def test_prompts_around_the_pieces_they_travel_in(n):
    """A prompt goes to the device in pieces of 896 tokens and its buffers are kept: the logits of one pass against the same
    tokens in two calls that share no piece boundary, with longer and shorter prompts in between."""
    import torch

    side = torch.cuda.Stream()
    dec = _decoder(max_ctx=2048)
    rng = np.random.default_rng(n)
    prompt = rng.integers(0, PCFG["vocab"], n).astype(np.int32)
    dec.prefill(prompt, stream=side.cuda_stream)
    one, first = dec.logits().copy(), dec.tokens(0, 1).copy()
    dec.prefill(rng.integers(0, PCFG["vocab"], 40).astype(np.int32))
    dec.prefill(rng.integers(0, PCFG["vocab"], 2000).astype(np.int32))
    dec.prefill(prompt[:500])
    dec.prefill(prompt[500:], start_pos=500, stream=side.cuda_stream)
    two = dec.logits().copy()
    assert np.abs(one - two).max() < 1e-2 * np.abs(one).max()
    dec.prefill(prompt)
    assert np.array_equal(dec.logits(), one) and np.array_equal(dec.tokens(0, 1), first)
