"""Correlations at the edges of a wave's rows and of the two block sizes."""

import numpy as np
import pytest
import torch

import calcir_amd as C
from calcir_amd import stages as S
from conftest import announce

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
PAIRS = ([(0, 0), (1, 1), (2, 2)], [(3, 3), (4, 4), (5, 5)], [(6, 6), (7, 7), (8, 8)],
         [(4, 3), (5, 3), (3, 4), (5, 4), (3, 5), (4, 5)])


@pytest.mark.parametrize("n", [1, 63, 64, 65, 257, 1023, 1024, 1025, 2101])
@pytest.mark.parametrize("nslot,pad", [(1, 0), (5, 3)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["fp32", "fp64"])
def test_correlation_edges(n, nslot, pad, dtype):
    announce("correlate n=%d nslot=%d %s" % (n, nslot, dtype))
    rng = np.random.default_rng(n + nslot)
    ncols = 9 * nslot
    sites = torch.from_numpy(rng.standard_normal((C.NSITE, n))).to(dtype)
    Y = torch.from_numpy(rng.standard_normal((n, 2 * ncols + pad))).to(dtype)
    Y[:, 2 * ncols:] = float("nan")  # the padding is not read
    got = S.correlate(sites.to(DEV), Y.to(DEV), nslot=nslot).numpy()
    M = sites[C.SITE_MU:C.SITE_MU + 9].double().numpy()
    Yc = Y[:, :ncols].double().numpy() + 1j * Y[:, ncols:2 * ncols].double().numpy()
    # one rounding per product (each below ~16 here), summed in 64 bits
    eps = 1.2e-7 if dtype == torch.float32 else 2.3e-16
    tol = 6 * 16 * eps * max(n, 16)
    for s in range(nslot):
        ir, a1, a2, a3 = (sum(M[b] @ Yc[:, 9 * s + a] for b, a in pr) for pr in PAIRS)
        ref = np.array([ir, (3 * a1 + a3 + 4 * a2) / 15, (2 * a1 - a3 + 6 * a2) / 30])
        assert np.abs(got[s] - ref).max() <= tol
