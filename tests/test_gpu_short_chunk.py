"""A last chunk shorter than the others, N >= 1024 (where batches of at most 16
matrices take the eigenpairs' correction): the results of one chunk."""

import functools

import numpy as np
import pytest

import calcir_amd as C
from calcir_amd.adjoint import LineshapeSession
from conftest import announce

pytestmark = pytest.mark.gpu
KEYS = ("tcf_ir", "tcf_vv", "tcf_vh", "sw")


def _params(prec, nframes, **kw):
    return C.default_params(species="H2O", model="tip4p2005", map=0, ntcfpoints=nframes - 4, nsamples=2,
                            origin_stride_frames=4, avef=3400.0, omegaStart=2800.0, omegaStop=4000.0, omegaStep=5,
                            nzeros=100 - nframes, t1=0.26, dt=0.010, precision=prec, **kw)


@functools.lru_cache(maxsize=None)
def _trajectory(nwater, nframes):
    return C.synth_trajectory(nwater, nframes, 40 + nwater)


@pytest.mark.parametrize("prec", ["fp32", "bf16x3"])
@pytest.mark.parametrize("nwater,nframes,chunk", [(512, 33, 17), (512, 36, 20), (520, 38, 23), (512, 40, 12)])
def test_short_last_chunk(nwater, nframes, chunk, prec):
    announce("short chunk nwater=%d frames=%d chunk=%d %s" % (nwater, nframes, chunk, prec))
    t = _trajectory(nwater, nframes)
    ref = C.run(_params(prec, nframes, chunk=nframes), *t)
    got = C.run(_params(prec, nframes, chunk=chunk), *t)
    # eigenvalues to 1e-6 of a spectrum of 1e3 cm^-1 over 0.4 ps: 1e-4 of a phase
    for k in KEYS:
        a, b = np.asarray(got[k]), np.asarray(ref[k])
        assert np.abs(a - b).max() <= 1e-4 * np.abs(b).max(), k


def test_gradient_with_a_short_last_chunk():
    announce("short chunk gradient")
    t = _trajectory(512, 33)
    out = []
    for chunk, store in ((33, 1), (17, 2)):
        s = LineshapeSession(_params("fp32", 33, chunk=chunk, adjoint_store=store), *t)
        f = np.asarray(s.forward())
        out.append((f, np.asarray(s.backward(np.cos(0.03 * np.arange(f.size)))) * np.asarray(s.coefs())))
    for a, b in zip(out[1], out[0]):
        assert np.abs(a - b).max() <= 1e-3 * np.abs(b).max()
