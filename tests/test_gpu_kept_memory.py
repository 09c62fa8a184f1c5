"""Device memory kept between runs: the same results from kept blocks and on
several threads, and no growth from run to run."""

import threading

import numpy as np
import pytest
import torch

import calcir_amd as C
from conftest import announce

pytestmark = pytest.mark.gpu
KEYS = ("tcf_ir", "tcf_vv", "tcf_vh", "sw")


def _job(waters, seed):
    xyz, box, times = C.synth_trajectory(waters, 12, seed)
    p = C.default_params(species="H2O", model="tip4p2005", map=0, ntcfpoints=6, nsamples=2, origin_stride_frames=4,
                         avef=3400.0, omegaStart=2800.0, omegaStop=4000.0, omegaStep=5, nzeros=58, t1=0.26, dt=0.010,
                         cutoff=0.7831, precision="fp32")
    return p, torch.from_numpy(xyz).to("cuda:0"), torch.from_numpy(box).to("cuda:0"), times


def test_runs_from_kept_blocks():
    announce("kept memory: sizes in turn")
    jobs = [_job(w, 300 + w) for w in (64, 200, 128, 240)]
    first = [C.run_device(*j) for j in jobs]
    free0 = torch.cuda.mem_get_info()[0]
    for _ in range(3):  # blocks of other sizes' runs, with their values in them
        for j, f in zip(jobs[::-1], first[::-1]):
            g = C.run_device(*j)
            for k in KEYS:
                assert np.abs(np.asarray(g[k]) - np.asarray(f[k])).max() <= 2e-5 * np.abs(np.asarray(f[k])).max(), k
    # bounded: one run's blocks at most are added to what is kept
    assert free0 - torch.cuda.mem_get_info()[0] < (1 << 30)


def test_runs_on_threads():
    announce("kept memory: threads")
    jobs = [_job(w, 500 + w) for w in (64, 100, 128, 150)]
    first = [C.run_device(*j) for j in jobs]
    out = [[None] * 3 for _ in jobs]

    def work(q):
        with torch.cuda.stream(torch.cuda.Stream()):
            for i in range(3):
                out[q][i] = C.run_device(*jobs[q])

    torch.cuda.synchronize()
    ts = [threading.Thread(target=work, args=(q,)) for q in range(len(jobs))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for q, f in enumerate(first):
        for g in out[q]:
            for k in KEYS:
                assert np.abs(np.asarray(g[k]) - np.asarray(f[k])).max() <= 2e-5 * np.abs(np.asarray(f[k])).max(), k
