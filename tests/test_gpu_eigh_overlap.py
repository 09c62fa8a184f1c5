"""Eigenvalues of FP32 Hamiltonians with a nearly overlapping pair of molecules
(a coupling of 1e5 cm^-1 beside bands of 1e3): the corrected ones are within
2e-8 of the largest (the correction is second order in the vectors' error, at
most 3e-5, and its products' error is 1e-5 of a residual below 1e-6), so the
band's are not drowned in the rounding of the pair's."""

import numpy as np
import pytest
import torch

import calcir_amd as C
from calcir_amd import stages as S
from conftest import announce

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n,batch", [(66, 3), (130, 2), (256, 3), (257, 2), (766, 18), (1023, 2), (1024, 2), (2081, 2)])
@pytest.mark.parametrize("prec", [C.PREC_FP32, C.PREC_BF16X3], ids=["fp32", "bf16x3"])
def test_overlapping_pair(n, batch, prec):
    announce("eigh overlap n=%d batch=%d prec=%d" % (n, batch, prec))
    rng = np.random.default_rng(n)
    H = rng.standard_normal((2, n, n)) * 3.0
    H = (H + np.transpose(H, (0, 2, 1))) / 2
    for b in range(2):
        H[b] += np.diag(rng.uniform(-400.0, 300.0, n))
        i, j = sorted(rng.choice(n, 2, replace=False))
        H[b, i, j] = H[b, j, i] = 1.0e5 * (1 if b else -1)
        H[b, i, :i] = H[b, :i, i] = H[b, i, :i] * 300.0  # its molecules' other couplings
    H = H.astype(np.float32)
    ld = (n + 3) // 4 * 4
    Hd = torch.zeros((batch, n, ld), device=DEV)
    Hd[:, :, :n] = torch.from_numpy(H[0]).to(DEV)
    Hd[batch - 1, :, :n] = torch.from_numpy(H[1]).to(DEV)
    w, V = S.eigh(Hd, n, prec=prec)
    for k, b in ((0, 0), (1, batch - 1)):
        wn = np.linalg.eigvalsh(H[k].astype(np.float64))
        assert np.abs(w[b].cpu().numpy() - wn).max() <= 2e-8 * np.abs(wn).max()
