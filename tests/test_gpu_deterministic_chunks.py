"""deterministic 1: the same bits whatever the chunk, on both sides of the sizes
and batches where the eigensolver's routes change."""

import numpy as np
import pytest

import calcir_amd as C
from conftest import announce

pytestmark = pytest.mark.gpu
KEYS = ("tcf_ir", "tcf_vv", "tcf_vh", "ftcf_ir", "ftcf_vv", "ftcf_vh", "sw")


@pytest.mark.parametrize("prec", ["fp32", "bf16x3"])
@pytest.mark.parametrize("nwater", [40, 128, 129, 511, 512, 1040])
def test_bits_do_not_depend_on_the_chunk(nwater, prec):
    announce("deterministic chunks nwater=%d %s" % (nwater, prec))
    nframes = 36 if nwater < 1000 else 20
    t = C.synth_trajectory(nwater, nframes, 552)
    ref = None
    for chunk in (nframes, 17, 12, 5):
        p = C.default_params(species="H2O", model="tip4p2005", map=0, ntcfpoints=nframes - 4, nsamples=2,
                             origin_stride_frames=4, avef=3400.0, omegaStart=2800.0, omegaStop=4000.0, omegaStep=5,
                             nzeros=100 - nframes, t1=0.26, dt=0.010, precision=prec, deterministic=1, chunk=chunk)
        got = C.run(p, *t)
        ref = ref or got
        for k in KEYS:
            assert np.array_equal(got[k], ref[k]), (chunk, k)
