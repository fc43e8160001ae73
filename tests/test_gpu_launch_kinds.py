"""Launches whose stepping kernel is not the default one keep its rate: tables
read from HBM instead of LDS, no energy loss, and a frame recorder. Times are
the best of five calls of 10^6 muons through the slab stack, in turn; results
are equal (test_gpu_parity, test_gpu_fp32, test_gpu_recorder)."""
import ctypes
import time

import numpy as np
import pytest

from parity import assert_parity
from test_gpu_recorder import grouped
from test_host_engine import build_host, run_host

import pumas_amd as pa
from pumas_amd import _abi
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


@pytest.mark.parametrize("precision", PRECISIONS)
@pytest.mark.parametrize("loss", [pa.Mode.CSDA, pa.Mode.DISABLED])
def test_recorder(gpu_standard, loss, precision):
    """A recorder of a hundred of the 10^6 histories."""
    ctx = W.slabs_forward_context(energy_loss=loss).replace(
        event=pa.Event.LIMIT_DISTANCE, limit_distance=500.0)
    rec = pa.Recorder(1 << 16, period=0, first_history=0, n_histories=100)
    plain, recorded = step_times(gpu_standard, [
        (ctx, dict(precision=precision)),
        (ctx, dict(precision=precision, recorder=rec))])
    assert rec.frames()[1] > 0
    assert recorded < 1.1 * plain


@pytest.mark.parametrize("options", [{}, dict(tail_del=-1),
                                     dict(lds_tables=-1),
                                     dict(max_steps=150)], ids=str)
@pytest.mark.parametrize("period", [0, 1, 7])
@pytest.mark.parametrize("forward", [True, False])
@pytest.mark.parametrize("loss", [pa.Mode.DISABLED, pa.Mode.CSDA,
                                  pa.Mode.MIXED, pa.Mode.STRAGGLED])
def test_frames_equal_host(gpu_standard, loss, forward, period, options):
    """Frames and final states of a batch whose middle half is recorded are
    those of the engine on the host, which steps a history at a time: steps,
    DELs, medium changes, and histories that a step limit ends."""
    make = W.slabs_forward_states if forward else W.slabs_backward_states
    ctx = (W.slabs_forward_context if forward else
           W.slabs_backward_context)(energy_loss=loss).replace(
        event=pa.Event.LIMIT_DISTANCE, limit_distance=600.0)
    desc = W.slabs_geometry()
    n, first, count, cap = 48, 12, 24, 1 << 20
    s = make(n, seed=31, **({} if forward else dict(kmax=50.0)))
    host = build_host()
    frames, k = np.zeros(cap, _abi.FRAME_DTYPE), ctypes.c_ulonglong(0)
    host.host_record(frames.ctypes.data, ctypes.addressof(k), cap, period,
                     first, count)
    host.host_set_max_steps(options.get("max_steps", 10000000))
    try:
        out = run_host(host, "standard_c005", ctx, desc, s, seed=6)
    finally:
        host.host_record(None, None, 0, 0, 0, 0)
        host.host_set_max_steps(10000000)
    ref = grouped(frames[:k.value])
    rec = pa.Recorder(cap, period=period, first_history=first,
                      n_histories=count)
    gpu = pa.transport(gpu_standard, ctx, pa.Geometry(gpu_standard, desc),
                       s.copy(), seed=6, recorder=rec, raise_errors=False,
                       **options)
    assert_parity(gpu, dict(zip(("final", "events", "media", "steps", "draws",
                                 "rc"), out)), 1e-12)
    f, total = rec.frames()
    assert total == len(ref) and 2 * count <= total <= cap
    f = grouped(f)
    for field in ("history", "event", "medium"):
        np.testing.assert_array_equal(f[field], ref[field])
    np.testing.assert_array_equal(f["state"]["charge"], ref["state"]["charge"])
    np.testing.assert_array_equal(f["state"]["decayed"],
                                  ref["state"]["decayed"])
    for field in ("energy", "distance", "grammage", "time", "weight"):
        np.testing.assert_allclose(f["state"][field], ref["state"][field],
                                   rtol=1e-12, atol=1e-300)
    for field in ("position", "direction"):
        np.testing.assert_allclose(f["state"][field], ref["state"][field],
                                   rtol=0, atol=1e-9)
