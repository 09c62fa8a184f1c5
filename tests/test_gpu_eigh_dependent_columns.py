"""Matrices with equal columns in their coupled part: what a panel leaves of them
falls by FP32's rounding from column to column, down to squares that underflow.
The reductions stay backward stable."""

import numpy as np
import pytest
import torch

import calcir_amd as C
from calcir_amd import stages as S
from conftest import announce

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n,batch", [(40, 2), (100, 2), (129, 2), (256, 2), (257, 2), (300, 2), (513, 2), (766, 2),
                                     (1023, 2), (1024, 2), (1100, 17), (2081, 2)])
@pytest.mark.parametrize("prec", [C.PREC_FP32, C.PREC_BF16X3], ids=["fp32", "bf16x3"])
def test_equal_columns(n, batch, prec):
    announce("eigh equal columns n=%d batch=%d prec=%d" % (n, batch, prec))
    H = np.diag(np.linspace(-300.0, 200.0, n)).astype(np.float32)
    H[:n // 2, :n // 2] += np.float32(7.0)
    Hd = torch.zeros((batch, n, (n + 3) // 4 * 4), device=DEV)
    Hd[:, :, :n] = torch.from_numpy(H).to(DEV)
    w, V = S.eigh(Hd, n, prec=prec)
    A = H.astype(np.float64)
    ref = np.linalg.eigvalsh(A)
    # backward error, and the vectors' bounds, as for the other sizes and routes
    tol = 50 * 6e-8 * np.sqrt(n)
    vtol = tol if prec == C.PREC_FP32 else 3e-4
    for b in (0, batch - 1):
        k, v = w[b].cpu().numpy(), V[b, :, :n].cpu().double().numpy()
        scale = np.abs(ref).max()
        assert np.abs(k - ref).max() <= tol * scale
        assert np.abs(A @ v - v * k).max() <= vtol * scale
        assert np.abs(v.T @ v - np.eye(n)).max() <= vtol
