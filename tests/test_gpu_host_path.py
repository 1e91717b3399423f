"""The native host path among Python's other threads and under torch's modes."""
import threading
import time

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from tcfp_amd import _hip
from tcfp_amd import kernels as K

pytestmark = pytest.mark.gpu


def test_other_threads_run_while_an_allocation_waits_for_the_gpu(dev):
    """With the process at its memory limit an output is made room for by
    freeing cached blocks, which waits for the GPU (here a spin of ~0.4 s);
    a counting thread goes on meanwhile."""
    t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda._sleep(1000)
    t0.record()
    torch.cuda._sleep(1_000_000)
    t1.record()
    torch.cuda.synchronize()
    cycles = int(1_000_000 * 400 / max(t0.elapsed_time(t1), 0.2))
    x = torch.zeros(1 << 14, 1 << 15, dtype=torch.bfloat16, device=dev)
    K.quantize_per_tensor(x[:8])  # (scratch and modules are there)
    torch.cuda.empty_cache()
    cached = [torch.empty(384 << 20, dtype=torch.uint8, device=dev) for _ in range(2)]
    del cached  # two blocks, neither large enough for the codes' 512 MiB
    ticks, stop = [], threading.Event()

    def count():
        while not stop.is_set():
            ticks.append(time.perf_counter())
            time.sleep(0.002)

    th = threading.Thread(target=count)
    try:
        torch.cuda.set_per_process_memory_fraction(
            (torch.cuda.memory_reserved() + (16 << 20)) / torch.cuda.mem_get_info()[1])
        th.start()
        torch.cuda._sleep(cycles)
        a = time.perf_counter()
        q, _ = K.quantize_per_tensor(x)
        b = time.perf_counter()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
        stop.set()
        if th.ident:
            th.join()
        torch.cuda.synchronize()
    during = sum(a < t < b for t in ticks)
    print(f"call took {b - a:.3f} s, {during} ticks of the other thread")
    assert b - a > 0.1, "the allocator did not wait: the test measures nothing"
    assert during > 20
    assert q.shape == x.shape


def test_threads_that_share_a_stream(dev):
    """Two-launch casts of two threads on one stream, whose partial maxima go
    through one scratch buffer: each thread's scale is its own tensor's."""
    xs = [torch.full((512, 512), float(v), device=dev) for v in (3.0, 50.0)]
    got = []

    def work(x):
        for _ in range(300):
            _, inv = K.quantize_per_tensor(x)
            got.append((inv, x))

    ths = [threading.Thread(target=work, args=(x,)) for x in xs]
    for t in ths:
        t.start()
    for t in ths:
        t.join()
    want = {id(x): K.quantize_per_tensor(x)[1].item() for x in xs}
    bad = [1 for inv, x in got if inv.item() != want[id(x)]]
    assert len(got) == 600 and not bad


class _Boom(Exception):
    pass


class _OnEmpty(TorchDispatchMode):
    """Calls `hook` ahead of every allocation."""

    def __init__(self, hook):
        super().__init__()
        self.hook = hook

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        if func is torch.ops.aten.empty.memory_format:
            self.hook(args[0])
        return func(*args, **(kwargs or {}))


def test_a_dispatch_modes_exception_keeps_its_type(dev):
    x = torch.randn(64, 64, device=dev)

    def hook(size):
        raise _Boom("no")

    with pytest.raises(_Boom, match="no"), _OnEmpty(hook):
        K.block_quantize_fp8(x, 64)
    assert K.block_quantize_fp8(x, 64)[0].shape == x.shape


def test_a_dispatch_mode_may_call_ops_while_the_scratch_is_allocated(dev):
    """The first call on a stream allocates its scratch; a mode's code that
    runs there may use the ops on the same stream."""
    x = torch.randn(512, 512, device=dev)
    nbytes = int(_hip.lib().tcfp_workspace_bytes())
    inner = []

    def hook(size):
        if list(size) == [nbytes] and not inner:
            inner.append(None)
            inner[0] = K.quantize_per_tensor(x)

    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(st):
        with _OnEmpty(hook):
            q, inv = K.quantize_per_tensor(x)
    st.synchronize()
    ref, rinv = K.quantize_per_tensor(x)
    torch.cuda.synchronize()
    assert torch.equal(q.view(torch.uint8), ref.view(torch.uint8)) and torch.equal(inv, rinv)
    if inner:  # (a pool stream that an earlier test has used has its scratch)
        assert torch.equal(inner[0][0].view(torch.uint8), ref.view(torch.uint8))
