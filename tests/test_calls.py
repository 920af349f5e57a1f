"""The native form of the short Python calls (csrc/calls.cpp) against the general way through ctypes, and what it does not take."""
import os
import subprocess
import sys

import numpy as np
import pytest


def test_calls_that_are_not_taken_go_the_general_way():
    import torch

    from yscv_amd import _calls, kernels, onnx_ops

    kernels.lib()
    host = torch.zeros(2, 64)
    assert _calls.int4_matmul(None, host, 64, 32) is None  # closed handle, host tensor
    assert _calls.int8_matmul(None, host, 64, 32, 0) is None
    assert _calls.dql_matmul(None, host, 64, 32) is None
    assert _calls.rms_norm(host, host[0], 1e-5) is None
    assert _calls.gqa(host, host, host, 1, 1) is None
    assert _calls.int4_matmul(None, None, 64, 32) is None and _calls.rms_norm(1, 2, 3) is None
    with pytest.raises(TypeError):  # the general way's errors
        onnx_ops.rms_norm(host, host[0], 1e-5)
    with pytest.raises(TypeError):
        onnx_ops.exec_grouped_query_attention(host[None], host[None], host[None], 1)
    with pytest.raises(TypeError):
        _calls.bind(1)


@pytest.mark.parametrize("module", ["None", "types.SimpleNamespace(torch_version=lambda: '0.0')", "types.SimpleNamespace()"])
def test_without_a_module_that_fits(module):
    """Not built, built for another torch, or an older build that does not say for which: the package is there all the same, and every call goes the general way."""
    code = f"""
import sys, types, warnings
warnings.simplefilter("ignore")
import yscv_amd
sys.modules["yscv_amd._calls"] = yscv_amd._calls = {module}
if yscv_amd._calls is None: del yscv_amd._calls
import torch
from yscv_amd import kernels as K, onnx_ops as O, short_calls
assert K.lib().abi_version() == 1 and short_calls.calls.rms_norm(1, 2, 3) is None
host = torch.zeros(2, 64)
for call, error in ((lambda: O.rms_norm(host, host[0], 1e-5), TypeError), (lambda: K.PackedI8B.matmul(types.SimpleNamespace(_h=None, _k=64, _n=2), host), AssertionError)):
    try:
        call()
    except error:
        continue
    raise SystemExit("no error")
"""
    run = subprocess.run([sys.executable, "-c", code], cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))), timeout=100)
    assert run.returncode == 0


@pytest.mark.gpu
def test_same_results_as_the_general_way():
    import torch

    from yscv_amd import kernels as K
    from yscv_amd import onnx_ops as O

    rng = np.random.default_rng(2)
    n, k = 48, 96
    w = K.PackedInt4Weight(rng.integers(0, 256, n * k // 2, dtype=np.uint8), rng.uniform(0.005, 0.02, n * k // 32).astype(np.float16), 32, n, k)
    for dtype in (torch.float32, torch.float16, torch.bfloat16):
        for shape in ((k,), (3, k), (2, 5, k)):
            x = torch.randn(shape, device="cuda").to(dtype)
            y = w.matmul(x)
            assert y.shape == (*shape[:-1], n) and y.dtype == dtype
            out = torch.empty_like(y)
            assert torch.equal(w.matmul(x, out=out), y)
            wide = torch.randn((*shape[:-1], 2 * k), device="cuda").to(dtype)[..., ::2]  # not contiguous
            assert torch.equal(w.matmul(wide), w.matmul(wide.contiguous()))
    with pytest.raises(K.capi.YscvHipError):  # no rows: a null pointer, refused
        w.matmul(torch.empty(0, k, device="cuda"))
    bm = rng.integers(-127, 128, (k, n), dtype=np.int8)
    b = K.pack_i8_b_for_matmul(bm, k, n)
    comp = torch.rand(n, device="cuda") * 0.01
    for dtype, zp in ((torch.uint8, 131), (torch.int8, -7)):
        a = torch.randint(0, 127, (9, k), device="cuda").to(dtype)
        assert torch.equal(b.matmul(a, a_zp=zp), b.matmul(a, a_zp=zp, out=torch.empty(9, n, device="cuda", dtype=torch.int32)))
        for lo, hi, odt in ((0, 255, torch.uint8), (-128, 127, torch.int8)):
            y = b.matmul_requant(a, zp, comp, 3.0, K.ROUND_HALF_AWAY, lo, hi)
            assert y.dtype == odt
            assert torch.equal(y, b.matmul_requant(a, zp, comp, 3.0, K.ROUND_HALF_AWAY, lo, hi, out=torch.empty_like(y)))
    with pytest.raises(K.capi.YscvHipError):  # refused by the library, by its status
        b.matmul(torch.zeros(1, k, device="cuda", dtype=torch.int8), a_zp=200)
    with pytest.raises(AssertionError):
        w.matmul(torch.zeros(1, k + 1, device="cuda"))
    pre = O.PrepackedI8B(torch.from_numpy(bm.astype(np.float32)).cuda())
    x = torch.randn(7, 2 * k, device="cuda")[:, ::2]
    for got, want in zip(O.exec_dql_matmul_integer(x.contiguous(), pre), O.exec_dql_matmul_integer(x, pre)):
        assert got.shape == want.shape and torch.equal(got, want)
    h, g = torch.randn(3, 4, 64, device="cuda"), torch.rand(64, device="cuda")
    assert torch.equal(O.rms_norm(h, g, 1e-5), O.rms_norm(h, g, np.float64(1e-5)))
    q, kv = torch.randn(2, 5, 128, device="cuda"), torch.randn(2, 9, 64, device="cuda")
    assert torch.equal(O.exec_grouped_query_attention(q, kv, kv, 4, 2), O.exec_grouped_query_attention(q.transpose(0, 1).contiguous().transpose(0, 1), kv, kv, 4, 2))
    w.close()
    with pytest.raises(K.capi.YscvHipError):
        w.matmul(torch.zeros(1, k, device="cuda"))


@pytest.mark.gpu
def test_other_threads_run_while_the_output_is_allocated():
    """Mapping memory for an output of 4 GiB takes 0.4 ms: a call that held the interpreter would stop the other thread for as long."""
    import threading
    import time

    import torch

    from yscv_amd import kernels as K

    m, n, k = 1 << 17, 8192, 64
    b = K.pack_i8_b_for_matmul(np.ones((k, n), np.int8), k, n)
    a = torch.ones(m, k, dtype=torch.uint8, device="cuda")
    b.matmul(a[:8])
    ticks, stop = [], threading.Event()

    def tick():
        while not stop.is_set():
            ticks.append(time.perf_counter())

    shares, interval = [], sys.getswitchinterval()
    sys.setswitchinterval(1e-5)  # (the time until the call has the interpreter back is no part of it)
    for _ in range(3):
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        ticks.clear()
        stop.clear()
        other = threading.Thread(target=tick)
        other.start()
        time.sleep(0.01)
        t0 = time.perf_counter()
        y = b.matmul(a)
        t1 = time.perf_counter()
        stop.set()
        other.join()
        inside = [t0] + [t for t in ticks if t0 < t < t1] + [t1]
        gap = max(q - p for p, q in zip(inside, inside[1:]))
        shares.append(gap / (t1 - t0))
        print(f"call {1e3 * (t1 - t0):.2f} ms, longest stop of the other thread {1e3 * gap:.2f} ms", flush=True)
        assert bool((y[-1] == k).all())
        del y
    sys.setswitchinterval(interval)
    assert min(shares) < 0.4


@pytest.mark.gpu
def test_modes_and_streams_are_seen():
    import torch
    from torch.utils._python_dispatch import TorchDispatchMode

    from yscv_amd import kernels as K

    rng = np.random.default_rng(4)
    n, k = 64, 64
    w = K.PackedInt4Weight(rng.integers(0, 256, n * k // 2, dtype=np.uint8), np.full(n * k // 32, 0.01, np.float16), 32, n, k)
    x = torch.randn(2, k, device="cuda")
    y = w.matmul(x)

    class Seen(TorchDispatchMode):
        names = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.names.append(str(func))
            return func(*args, **(kwargs or {}))

    with Seen():
        assert torch.equal(w.matmul(x), y)
    assert any("new_empty" in s for s in Seen.names)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        graph.capture_begin()
        z = w.matmul(x)  # reaches the capturing stream, the current one
        graph.capture_end()
    for _ in range(3):
        z.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(z, y)
    with pytest.raises(RuntimeError):  # a batched tensor has no storage
        torch.vmap(w.matmul)(x)


@pytest.mark.gpu
@pytest.mark.parametrize("call", ["O.rms_norm(x, g, 1e-5)", "O.exec_grouped_query_attention(x, x, x, 1, 1)"])
def test_the_first_call_of_a_process(call):
    """Nothing has loaded the library yet: the call goes the general way."""
    code = ("import torch; from yscv_amd import onnx_ops as O; x, g = torch.ones(1, 4, 64, device='cuda'), torch.ones(64, device='cuda'); "
            "y = " + call + "; z = " + call + "; torch.cuda.synchronize(); assert bool(((y - 1).abs() < 1e-3).all()) and bool((y == z).all())")
    run = subprocess.run([sys.executable, "-c", code], cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))), timeout=100)
    assert run.returncode == 0
