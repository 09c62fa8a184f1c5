"""Dense to band at the sizes where the panel kernel's rows per thread change,
with panels that are zero below the band already."""

import numpy as np
import pytest
import torch

import calcir_amd as C
from calcir_amd import stages as S
from conftest import announce

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# the first panel has n - 32 rows, 512 per register row; 17 matrices of
# N >= 1024 take the route without a correction of the eigenpairs
@pytest.mark.parametrize("n,batch,band", [(544, 2, 0), (545, 2, 0), (1056, 17, 0), (1057, 17, 0), (1063, 17, 20),
                                          (1568, 17, 0), (1569, 17, 0), (2080, 17, 0), (2079, 17, 33), (2081, 2, 0),
                                          (2592, 2, 0), (2593, 2, 31), (3104, 2, 0), (3105, 2, 0)])
def test_two_stage_at_panel_edges(n, batch, band):
    announce("band panels n=%d batch=%d band=%d" % (n, batch, band))
    rng = np.random.default_rng(n)
    # (all matrices on the card; the first and the last are compared)
    H = rng.standard_normal((2, n, n)) * 3.0
    H = (H + np.transpose(H, (0, 2, 1))) / 2
    if band:
        i = np.arange(n)
        H *= np.abs(i[:, None] - i) < band
    for b in range(2):
        H[b] += np.diag(rng.uniform(-400.0, 300.0, n))
    H = H.astype(np.float32)
    ld = (n + 3) // 4 * 4
    Hd = torch.zeros((batch, n, ld), device=DEV)
    Hd[:, :, :n] = torch.from_numpy(H[0]).to(DEV)
    Hd[batch - 1, :, :n] = torch.from_numpy(H[1]).to(DEV)
    w, V = S.eigh(Hd, n, prec=C.PREC_FP32)
    eps = 6e-8
    for k, b in ((0, 0), (1, batch - 1)):
        wb, Vb = w[b].cpu().numpy(), V[b].cpu().double().numpy()[:, :n]
        Hb = H[k].astype(np.float64)
        wn = np.linalg.eigvalsh(Hb)
        scale = np.abs(wn).max()
        # backward error of the reduction, as for the other two-stage sizes
        assert np.abs(wb - wn).max() <= 50 * eps * scale * np.sqrt(n)
        assert np.abs(Hb @ Vb - Vb * wb).max() / scale < 50 * eps * np.sqrt(n)
        assert np.abs(Vb.T @ Vb - np.eye(n)).max() < 50 * eps * np.sqrt(n)
