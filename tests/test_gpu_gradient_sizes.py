"""The gradient's products at box sizes on either side of their tiles: FP32
against FP64."""

import numpy as np
import pytest

import calcir_amd as C
from calcir_amd.adjoint import LineshapeSession
from conftest import announce

pytestmark = pytest.mark.gpu

KW = dict(species="H2O", model="tip4p2005", map=0, ntcfpoints=10, nsamples=4, origin_stride_frames=2, avef=3400.0, omegaStart=2800.0,
          omegaStop=4000.0, omegaStep=5, nzeros=246, t1=0.26, dt=0.010)


# seeds without close contacts (whose FP32 rounding alone moves the spectrum)
@pytest.mark.parametrize("waters,seed", [(48, 933), (49, 920), (63, 940), (64, 919), (65, 952), (81, 953)])
@pytest.mark.parametrize("prec", ["fp32", "bf16x3"])
def test_gradient_at_tile_edges(waters, seed, prec):
    announce("gradient sizes waters=%d %s" % (waters, prec))
    xyz, box, times = C.synth_trajectory(waters, 18, seed)
    out = {}
    for q in ("fp64", prec):
        sess = LineshapeSession(C.default_params(precision=q, **KW), xyz, box, times)
        f = np.asarray(sess.forward())
        k = np.arange(f.size)
        g = np.cos(0.03 * k) * np.exp(-k / 60.0)
        out[q] = np.asarray(sess.backward(g)) * np.asarray(sess.coefs())
    # the single-precision forward's error, as in the gradient's other tests
    assert np.abs(out[prec] - out["fp64"]).max() <= 1e-3 * np.abs(out["fp64"]).max()
