"""Host side of a call: the pinned memory of its results, and what it waits
for."""
import ctypes
import os
import threading
import time

import pytest

import pumas_amd as pa
from pumas_amd import workloads as W

pytestmark = pytest.mark.gpu


def _buffers(n):
    """The pinned buffers of `n` threads that are alive together, once the
    threads have ended (joined, and gone from the process)."""
    f = pa.library()._Z9pg_pinnedm  # pg_pinned(size_t), status.h
    f.argtypes, f.restype = [ctypes.c_size_t], ctypes.c_void_p
    out, barrier = [], threading.Barrier(n)

    def run():
        p = f(256)
        out.append((threading.get_native_id(), p, f(256), f(1 << 20)))
        barrier.wait(30)

    threads = [threading.Thread(target=run) for _ in range(n)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    end = time.monotonic() + 30
    while any(os.path.exists(f"/proc/self/task/{t}") for t, *_ in out):
        assert time.monotonic() < end
        time.sleep(0.01)
    for _, p, again, large in out:
        assert p and again == p and large is None
    return [p for _, p, *_ in out]


def test_pinned_buffers_pass_between_threads(gpu_standard):
    """Threads alive together have a buffer each; those of ended threads are
    still allocated and serve the next threads, up to 16 of them."""
    flags = ctypes.c_uint()

    def allocated(p):
        lib = pa.library()
        rc = lib.hipHostGetFlags(ctypes.byref(flags), ctypes.c_void_p(p))
        lib.hipGetLastError()  # not left for the next call to report
        return rc == 0
    first = _buffers(4)
    assert len(set(first)) == 4
    assert all(allocated(p) for p in first)
    assert set(_buffers(2)) <= set(first)
    many = _buffers(24)
    assert len(set(many)) == 24
    assert sum(allocated(p) for p in many) == 16


def test_empty_batch_waits_for_the_stream(gpu_standard):
    """A call returns with its stream's work done, an empty batch's too."""
    import torch
    geom = pa.Geometry(gpu_standard, W.slabs_geometry())
    ctx = W.slabs_forward_context()
    a = torch.randn(4096, 4096, device="cuda")
    stream = torch.cuda.Stream()
    pa.transport_device(gpu_standard, ctx, geom, 0, 0,
                        stream=stream.cuda_stream)
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        for _ in range(200):
            b = a @ a
    assert not stream.query()
    pa.transport_device(gpu_standard, ctx, geom, 0, 0,
                        stream=stream.cuda_stream)
    assert stream.query()
    del b
