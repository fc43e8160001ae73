"""Host side of a call: what it waits for."""
import pytest

import pumas_amd as pa
from pumas_amd import workloads as W

pytestmark = pytest.mark.gpu


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
