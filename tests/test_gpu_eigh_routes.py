"""The eigensolver's routes at the sizes where they change: FP32 batches of any
size in two stages with the eigenpairs corrected afterwards (few or small
matrices), FP64 batches on either side of the whole-GPU rule."""

import numpy as np
import pytest
import torch

import calcir_amd as C
from calcir_amd import stages as S
from conftest import announce

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _matrices(n, batch, seed):
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((batch, n, n)) * 3.0
    H = (a + np.transpose(a, (0, 2, 1))) / 2
    for b in range(batch):
        d = rng.uniform(-400.0, 300.0, n)
        d[rng.integers(n)] -= 1500.0  # a strong-field outlier
        if b == 0 and n > 8:  # an uncoupled pair with equal frequencies
            H[b, :2] = H[b, :, :2] = 0.0
            d[0] = d[1] = 17.0
        H[b] += np.diag(d)
    return H


@pytest.mark.parametrize("n,batch", [(449, 1), (512, 3), (639, 17), (1023, 2), (1024, 16), (1100, 1), (2048, 2)])
@pytest.mark.parametrize("prec", [C.PREC_FP32, C.PREC_BF16X3], ids=["fp32", "bf16x3"])
def test_corrected_two_stage_eigenpairs(n, batch, prec):
    announce("eigh routes n=%d batch=%d prec=%d" % (n, batch, prec))
    H = _matrices(n, batch, n + batch).astype(np.float32)
    ld = (n + 3) // 4 * 4 + 4
    Hd = np.zeros((batch, n, ld), np.float32)
    Hd[:, :, :n] = H
    for b in range(batch):  # the triangle below the diagonal is not read
        Hd[b, :, :n][np.tril_indices(n, -1)] = 5.0e3
    w, V = S.eigh(torch.from_numpy(Hd).to(DEV), n, prec=prec)
    w, V = w.cpu().numpy(), V.cpu().double().numpy()[:, :, :n]
    eps = 6e-8
    vtol = 50 * eps * np.sqrt(n) if prec == C.PREC_FP32 else 3e-4
    for b in {0, batch - 1}:
        Hb = H[b].astype(np.float64)
        wn = np.linalg.eigvalsh(Hb)
        scale = np.abs(wn).max()
        assert np.all(np.diff(w[b]) >= 0)
        # the corrected eigenvalues carry the rounding of one FP32 product,
        # a few eps of the couplings' norm (about 3 sqrt(n) sqrt(2) here) and
        # of the FP32 diagonal, against 50 eps sqrt(n) scale uncorrected
        assert np.abs(w[b] - wn).max() <= 8 * eps * scale, np.abs(w[b] - wn).max() / scale
        assert np.abs(Hb @ V[b] - V[b] * w[b]).max() / scale < vtol
        assert np.abs(V[b].T @ V[b] - np.eye(n)).max() < vtol


@pytest.mark.parametrize("n,batch", [(511, 1), (512, 1), (512, 2), (600, 3)])
def test_fp64_routes(n, batch):
    announce("eigh fp64 routes n=%d batch=%d" % (n, batch))
    H = _matrices(n, batch, 7 * n + batch)
    ld = (n + 3) // 4 * 4
    Hd = np.zeros((batch, n, ld))
    Hd[:, :, :n] = H
    w, V = S.eigh(torch.from_numpy(Hd).to(DEV), n)
    w, V = w.cpu().numpy(), V.cpu().numpy()[:, :, :n]
    for b in {0, batch - 1}:
        wn = np.linalg.eigvalsh(H[b])
        scale, eps = np.abs(wn).max(), 2.2e-16
        assert np.abs(w[b] - wn).max() <= 50 * eps * scale * np.sqrt(n)
        assert np.abs(H[b] @ V[b] - V[b] * w[b]).max() / scale < 50 * eps * np.sqrt(n)
        # inverse iteration: eps ||T|| / gap, as in the whole-GPU path's test
        assert np.abs(V[b].T @ V[b] - np.eye(n)).max() < 2000 * eps * np.sqrt(n)
