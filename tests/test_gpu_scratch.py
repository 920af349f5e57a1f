"""Scratch blocks the library keeps per stream: calls of growing and shrinking size on more streams than there are
blocks, from several threads on one stream, and inside a captured graph give what they give one at a time."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _weight(K, rng, n, k, g=64):
    return K.PackedInt4Weight(rng.integers(0, 256, n * k // 2, dtype=np.uint8), rng.uniform(0.005, 0.02, n * (k // g)).astype(np.float16),
                              g, n, k, nibble_format=K.NIBBLE_UNSIGNED)


def test_more_streams_than_blocks_and_growing_requests():
    import torch

    from yscv_amd import kernels as K

    rng = np.random.default_rng(1)
    w = _weight(K, rng, 208, 960)  # bf16 rows above 16 are prepared in the scratch, and K is cut into parts there
    xs = [torch.from_numpy(rng.standard_normal((m, 960)).astype(np.float32)).bfloat16().cuda() for m in (3, 700, 40, 5000, 77, 1, 300, 20, 64, 9, 2500, 130)]
    want = [w.matmul(x, out_dtype=torch.float32).clone() for x in xs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(11)]
    got = []
    for rnd in range(3):
        for i, x in enumerate(xs):
            with torch.cuda.stream(streams[(i * 5 + rnd) % len(streams)]):
                got.append((i, w.matmul(x, out_dtype=torch.float32)))
    torch.cuda.synchronize()
    for i, y in got:
        assert torch.equal(y, want[i]), i


def test_threads_on_one_stream():
    import torch

    from yscv_amd import kernels as K

    rng = np.random.default_rng(2)
    w = _weight(K, rng, 272, 1344)
    xs = [torch.from_numpy(rng.standard_normal((50 + 30 * t, 1344)).astype(np.float32)).bfloat16().cuda() for t in range(4)]
    want = [w.matmul(x, out_dtype=torch.float32).clone() for x in xs]
    torch.cuda.synchronize()
    got = [[] for _ in xs]

    def worker(t):
        for _ in range(50):
            got[t].append(w.matmul(xs[t], out_dtype=torch.float32))

    threads = [threading.Thread(target=worker, args=(t,)) for t in range(len(xs))]
    for th in threads:
        th.start()
    for th in threads:
        th.join(timeout=60)
    assert not any(th.is_alive() for th in threads)
    torch.cuda.synchronize()
    for t, ys in enumerate(got):
        assert len(ys) == 50 and all(torch.equal(y, want[t]) for y in ys), t


def test_captured_call_keeps_its_own_memory():
    import torch

    from yscv_amd import kernels as K

    rng = np.random.default_rng(3)
    w = _weight(K, rng, 208, 960)
    x = torch.from_numpy(rng.standard_normal((90, 960)).astype(np.float32)).bfloat16().cuda()
    other = torch.from_numpy(rng.standard_normal((4000, 960)).astype(np.float32)).bfloat16().cuda()
    want = w.matmul(x, out_dtype=torch.float32).clone()
    out = torch.empty_like(want)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        w.matmul(x, out=out)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=side):
            w.matmul(x, out=out)
    for _ in range(4):
        out.zero_()
        torch.cuda.synchronize()
        g.replay()
        w.matmul(other)  # another call's scratch between the replays
        torch.cuda.synchronize()
        assert torch.equal(out, want)


@pytest.mark.parametrize("where", ["used before", "new", "default", "growing"])
def test_a_call_beside_a_capture_of_another_stream(where):
    """Calls on one stream while another is captured (torch's default mode watches the whole process for calls that may not
    happen meanwhile): they run, and the capture goes on."""
    import ctypes as C

    import torch

    from yscv_amd import BF16, kernels as K, lib

    rng = np.random.default_rng(4)
    w = _weight(K, rng, 256, 512)
    x = torch.from_numpy(rng.standard_normal((24, 512)).astype(np.float32)).bfloat16().cuda()
    want = w.matmul(x)
    got, z = torch.zeros_like(want), torch.zeros(4, device="cuda")
    captured, other = torch.cuda.Stream(), torch.cuda.default_stream() if where == "default" else torch.cuda.Stream()
    long_x = torch.from_numpy(rng.standard_normal((9000, 512)).astype(np.float32)).bfloat16().cuda()
    long_want = w.matmul(long_x)
    long_got = torch.zeros_like(long_want)

    def call_long():
        lib().int4_matmul(w._h, C.c_void_p(long_x.data_ptr()), BF16, C.c_void_p(long_got.data_ptr()), BF16, C.c_size_t(9000),
                          C.c_void_p(other.cuda_stream))

    def call():
        lib().int4_matmul(w._h, C.c_void_p(x.data_ptr()), BF16, C.c_void_p(got.data_ptr()), BF16, C.c_size_t(24), C.c_void_p(other.cuda_stream))

    if where != "new":
        call()
    torch.cuda.synchronize()
    got.zero_()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=captured):
        z += 1
        for _ in range(3):
            call()
        if where == "growing":
            call_long()  # more than the block holds
    g.replay()
    torch.cuda.synchronize()
    assert where != "growing" or torch.equal(long_got, long_want)
    assert z.tolist() == [1.0] * 4 and torch.equal(got, want)
