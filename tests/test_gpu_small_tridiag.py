"""The register-resident reduction of small matrices at the edges of its
variants, reading one triangle only."""

import numpy as np
import pytest
import torch

from calcir_amd import stages as S
from conftest import announce

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n", [1, 2, 3, 16, 31, 33, 64, 127, 128, 129, 160, 191, 192, 193, 224, 255, 256, 257])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["fp32", "fp64"])
def test_small_eigenpairs(n, dtype):
    batch = 3
    announce("small tridiag n=%d %s" % (n, dtype))
    rng = np.random.default_rng(n)
    H = rng.standard_normal((batch, n, n)) * 3.0
    H = (H + np.transpose(H, (0, 2, 1))) / 2
    for b in range(batch):
        H[b] += np.diag(rng.uniform(-400.0, 300.0, n))
    if n > 8:
        H[1] = np.diag(np.diag(H[1]))  # nothing to annihilate
        H[2, 3:, :3] = H[2, :3, 3:] = 0.0  # two uncoupled blocks
    H = H.astype(np.float32 if dtype == torch.float32 else np.float64)
    ld = (n + 3) // 4 * 4 + 4
    Hd = np.full((batch, n, ld), 7.0e3, H.dtype)  # (finite padding, which is not read)
    Hd[:, :, :n] = H
    for b in range(batch):  # the other triangle is not read either
        Hd[b, :, :n][np.tril_indices(n, -1)] = -9.0e3
    w, V = S.eigh(torch.from_numpy(Hd).to(DEV), n)
    w, V = w.cpu().numpy(), V.cpu().double().numpy()[:, :, :n]
    eps = 6e-8 if dtype == torch.float32 else 1.2e-16
    for b in range(batch):
        Hb = H[b].astype(np.float64)
        wn = np.linalg.eigvalsh(Hb)
        scale = np.abs(wn).max()
        # backward stable: a modest multiple of eps sqrt(n) ||H||, as for the
        # other sizes; orthogonality as inverse iteration leaves it
        assert np.abs(w[b] - wn).max() <= 50 * eps * scale * np.sqrt(n)
        assert np.abs(Hb @ V[b] - V[b] * w[b]).max() / scale < 50 * eps * np.sqrt(n)
        assert np.abs(V[b].T @ V[b] - np.eye(n)).max() < (50 if eps > 1e-10 else 2000) * eps * np.sqrt(n)
