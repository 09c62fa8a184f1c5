"""Device memory kept between runs: no growth over rounds, given back on request
and by run_many, no obstacle to jobs that need it, and no use of a stream that
is gone."""

import ctypes

import numpy as np
import pytest
import torch

import calcir_amd as C
from calcir_amd.adjoint import LineshapeSession
from conftest import announce

pytestmark = pytest.mark.gpu
MB = 1 << 20
KEYS = ("tcf_ir", "tcf_vv", "tcf_vh", "sw")


def _params(points, **kw):
    return C.default_params(species="H2O", model="tip4p2005", map=0, ntcfpoints=points, nsamples=2, origin_stride_frames=2,
                            avef=3400.0, omegaStart=2800.0, omegaStop=4000.0, omegaStep=5, nzeros=2 * points, t1=0.26,
                            dt=0.010, cutoff=0.7831, precision="fp32", **kw)


def _device_job(waters, frames, seed):
    xyz, box, times = C.synth_trajectory(waters, frames, seed)
    return _params(frames - 2), torch.from_numpy(xyz).to("cuda:0"), torch.from_numpy(box).to("cuda:0"), times


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_no_growth_over_rounds():
    announce("kept memory limits: rounds")
    # at least a gigabyte a round (H, V and work space: over 20 MB a frame)
    jobs = [_device_job(w, 30, 900 + w) for w in (300, 384, 340)]
    for _ in range(2):
        for j in jobs:
            C.run_device(*j)
    free0 = _free()
    for _ in range(4):
        for j in jobs:
            C.run_device(*j)
    assert free0 - _free() < 256 * MB


def test_given_back_on_request_and_by_run_many():
    announce("kept memory limits: given back")
    job = _device_job(384, 40, 77)
    C.run_device(*job)
    C.release_memory()
    free0 = _free()
    C.run_device(*job)
    assert free0 - _free() > 256 * MB  # kept (over 20 MB a frame)
    C.release_memory()
    assert free0 - _free() < 64 * MB
    C.run_device(*job)
    xyz, box, times = C.synth_trajectory(64, 12, 5)
    C.run_many([(_params(10), xyz, box, times)])
    assert free0 - _free() < 64 * MB


def test_jobs_get_what_is_kept():
    announce("kept memory limits: jobs that need the kept memory")
    big, small = _device_job(512, 200, 31), C.synth_trajectory(512, 120, 32)
    p = _params(118)
    ref = C.run_many([(p,) + small])[0]  # about 4 GB
    C.run_device(*big)                   # keeps more than that
    # all but 2 GB of what is free taken by another user of the device
    hold = torch.empty(max(0, _free() - 2048 * MB), dtype=torch.uint8, device="cuda:0")
    try:
        got = C.run_many([(p,) + small])[0]
        alone = C.run(p, *small)
    finally:
        del hold
        torch.cuda.empty_cache()
    for k in KEYS:
        for r in (got, alone):
            assert np.abs(np.asarray(r[k]) - np.asarray(ref[k])).max() <= 2e-5 * np.abs(np.asarray(ref[k])).max(), k


def test_context_outlives_its_stream():
    announce("kept memory limits: stream destroyed before the context")
    L = C.lib()
    L.hipStreamCreate.argtypes, L.hipStreamDestroy.argtypes = [ctypes.c_void_p], [ctypes.c_void_p]
    xyz, box, times = C.synth_trajectory(100, 12, 9)
    p = _params(10)
    stream, ctx = ctypes.c_void_p(), ctypes.c_void_p()
    assert L.hipStreamCreate(ctypes.byref(stream)) == 0
    C.check(L.cir_create(ctypes.byref(p), xyz.shape[1], stream, ctypes.byref(ctx)))
    f = np.zeros(p.ntcfpoints + p.nzeros)
    C.check(L.cir_forward_ls(ctx, xyz.shape[0], xyz.ctypes.data, box.ctypes.data, times.ctypes.data, f.ctypes.data))
    torch.cuda.synchronize()
    assert L.hipStreamDestroy(stream) == 0
    L.cir_destroy(ctx)  # its kept buffers are freed without the stream
    s = LineshapeSession(p, xyz, box, times)
    g = np.asarray(s.forward())
    assert np.abs(f - g).max() <= 2e-5 * np.abs(g).max()
