"""The bulge-chasing reflectors on the eigenvectors for each slab width, at
ragged slabs and at sizes with fewer groups of sweeps than waves."""

import numpy as np
import pytest
import torch

import calcir_amd as C
from calcir_amd import stages as S
from conftest import announce

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# slabs of 64 columns from ceil(n / 64) batch = 512 on (split BF16), of 32 from
# ceil(n / 32) batch = 512 on, else of 16; 12 waves of one 16-sweep group each
@pytest.mark.parametrize("n,batch", [(66, 1), (67, 300), (97, 257), (130, 103), (191, 200), (205, 7), (449, 64),
                                     (512, 32), (513, 31), (577, 52)])
@pytest.mark.parametrize("prec", [C.PREC_FP32, C.PREC_BF16X3], ids=["fp32", "bf16x3"])
def test_two_stage_slabs(n, batch, prec, monkeypatch):
    announce("q2 slabs n=%d batch=%d prec=%d" % (n, batch, prec))
    monkeypatch.setenv("CIR_EIGH_STAGES", "2")
    rng = np.random.default_rng(n + batch)
    H = rng.standard_normal((3, n, n)) * 3.0
    H = (H + np.transpose(H, (0, 2, 1))) / 2
    for b in range(3):
        H[b] += np.diag(rng.uniform(-400.0, 300.0, n))
    H = H.astype(np.float32)
    ld = (n + 3) // 4 * 4
    Hd = torch.zeros((batch, n, ld), device=DEV)
    which = np.zeros(batch, int)  # the middle and the last matrix differ from the others
    which[batch // 2], which[batch - 1] = 1, 2
    for b in range(batch):
        Hd[b, :, :n] = torch.from_numpy(H[which[b]])
    w, V = S.eigh(Hd, n, prec=prec)
    eps = 6e-8
    vtol = 50 * eps * np.sqrt(n) if prec == C.PREC_FP32 else 3e-4
    for b in {0, batch // 2, batch - 1}:
        wb, Vb = w[b].cpu().numpy(), V[b].cpu().double().numpy()[:, :n]
        Hb = H[which[b]].astype(np.float64)
        wn = np.linalg.eigvalsh(Hb)
        scale = np.abs(wn).max()
        assert np.abs(wb - wn).max() <= 50 * eps * scale * np.sqrt(n)
        assert np.abs(Hb @ Vb - Vb * wb).max() / scale < vtol
        assert np.abs(Vb.T @ Vb - np.eye(n)).max() < vtol
    # equal matrices, equal columns
    same = torch.from_numpy(which == 0).to(DEV)
    assert bool((V[same] == V[0]).all())
