"""FP32 matrices at the ends of the scales that their squares allow: eigenvalues
within the reductions' backward error, a matrix of zeros included."""

import numpy as np
import pytest
import torch

import calcir_amd as C
from calcir_amd import stages as S
from conftest import announce

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# (below 1 the whole spectrum is one cluster of the inverse iteration, solved one
# vector after the other: small sizes)
@pytest.mark.parametrize("n,scale", [(n, s) for n in (1, 2, 5, 40, 160, 257) for s in (0.0, 1e-18, 1e-12, 1.0, 1e16)] +
                         [(600, 1e16), (1023, 1e12)])
@pytest.mark.parametrize("prec", [C.PREC_FP32, C.PREC_BF16X3], ids=["fp32", "bf16x3"])
def test_eigenvalues_at_any_scale(n, scale, prec):
    announce("eigh scales n=%d scale=%g prec=%d" % (n, scale, prec))
    a = np.random.default_rng(n).standard_normal((n, n))
    H = ((a + a.T) / 2 * scale).astype(np.float32)
    Hd = torch.zeros((2, n, (n + 3) // 4 * 4), device=DEV)
    Hd[:, :, :n] = torch.from_numpy(H).to(DEV)
    w, V = S.eigh(Hd, n, prec=prec)
    ref = np.linalg.eigvalsh(H.astype(np.float64))
    for b in range(2):
        got = w[b].cpu().numpy()
        # (zeros: at most the smallest normal number that pads the bracket)
        assert np.abs(got - ref).max() <= 50 * 6e-8 * np.sqrt(n) * np.abs(ref).max() + 1e-307
        assert np.all(np.diff(got) >= 0)
