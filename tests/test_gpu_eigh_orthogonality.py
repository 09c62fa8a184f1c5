"""Corrected eigenvectors are orthogonal to FP32's rounding in split BF16 too:
each column scaled to length one and rounded twice (2 x 1.5 eps of a product of
two columns at most, 2e-7), the first-order rotations' second order (2 / 2048^2
at most, 5e-7) and the rounding of V^T V formed in runs of 128 rows (1e-7)."""

import numpy as np
import pytest
import torch

import calcir_amd as C
from calcir_amd import stages as S
from cases import frames
from conftest import announce

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# every size below 1024, batches of at most 16 up to 2080, every size above it
@pytest.mark.parametrize("nwater,batch", [(1, 3), (17, 2), (64, 17), (128, 5), (129, 2), (200, 20), (383, 17), (511, 2),
                                          (512, 16), (700, 2), (1041, 2)])
@pytest.mark.parametrize("prec", [C.PREC_FP32, C.PREC_BF16X3], ids=["fp32", "bf16x3"])
def test_corrected_eigenvectors_are_orthogonal(nwater, batch, prec):
    announce("eigh orthogonality nwater=%d batch=%d prec=%d" % (nwater, batch, prec))
    xyz, box, _ = frames(nwater, batch, 700 + nwater)
    b = torch.from_numpy(box.copy()).to(DEV)
    sg = S.eproj_sites(torch.from_numpy(xyz.copy()).to(DEV), b, dtype=torch.float32)
    H = S.hamiltonian(sg, b, avef=3400.0)
    n = 2 * nwater
    Hd = H[batch - 1, :, :n].double()
    w, V = S.eigh(H, n, prec=prec)
    v = V[batch - 1, :, :n].double()
    assert float((v.T @ v - torch.eye(n, dtype=torch.float64, device=DEV)).abs().max()) <= 1e-6
    # and still eigenvectors: as close as the routes' other tests ask of FP32
    res = (Hd @ v - v * w[batch - 1]).abs().max() / w[batch - 1].abs().max()
    assert float(res) < 50 * 6e-8 * np.sqrt(n)
