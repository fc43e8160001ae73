"""Launches whose stepping kernel is not the default one keep its rate: tables
read from HBM instead of LDS, no energy loss, and a frame recorder. Times are
the best of five calls of 10^6 muons through the slab stack, in turn; results
are equal (test_gpu_parity, test_gpu_fp32, test_gpu_recorder)."""
import time

import numpy as np
import pytest

import pumas_amd as pa
from pumas_amd import workloads as W

pytestmark = pytest.mark.gpu

N = 1000003
PRECISIONS = [pa.Precision.FP64, pa.Precision.FP32_BULK]


def step_times(physics, calls):
    """Seconds per step of each (context, options)."""
    import torch
    first = torch.from_numpy(W.slabs_forward_states(N, seed=3).view(
        np.float64).reshape(-1, 13)).cuda()
    work = torch.empty_like(first)
    geom = pa.Geometry(physics, W.slabs_geometry())
    best = [np.inf] * len(calls)
    for rep in range(6):
        for k, (ctx, options) in enumerate(calls):
            work.copy_(first)
            torch.cuda.synchronize()
            t = time.perf_counter()
            st = pa.transport_device(physics, ctx, geom, work.data_ptr(), N,
                                     seed=5, **options)
            t = (time.perf_counter() - t) / st.steps
            if rep > 0:
                best[k] = min(best[k], t)
    print("ps per step:", [round(1e12 * b, 1) for b in best], flush=True)
    return best


@pytest.mark.parametrize("precision", PRECISIONS)
def test_tables_in_hbm(gpu_standard, precision):
    ctx = W.slabs_forward_context(energy_loss=pa.Mode.CSDA)
    lds, hbm = step_times(gpu_standard, [
        (ctx, dict(precision=precision)),
        (ctx, dict(precision=precision, lds_tables=-1))])
    assert hbm < 1.2 * lds


@pytest.mark.parametrize("precision", PRECISIONS)
def test_no_energy_loss(gpu_standard, precision):
    """Without energy loss a step does less than with the CSDA."""
    csda = W.slabs_forward_context(energy_loss=pa.Mode.CSDA)
    none = W.slabs_forward_context(energy_loss=pa.Mode.DISABLED).replace(
        event=pa.Event.LIMIT_DISTANCE, limit_distance=500.0)
    a, b = step_times(gpu_standard, [(csda, dict(precision=precision)),
                                     (none, dict(precision=precision))])
    assert b < 1.05 * a
