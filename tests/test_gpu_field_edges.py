"""Field and Hamiltonian kernels at the sizes where their splits can go wrong:
chromophores that do not fill a workgroup, neighbour lists that are flushed
more than once (every molecule inside the cutoff) or never (none), more
molecules than one staged tile, tiles of H cut by N and by the leading
dimension."""

import numpy as np
import pytest
import torch

import calcir_amd as C
import oracle_lib as O
from calcir_amd import stages as S
from cases import frames
from conftest import announce

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("nwater,cutoff", [(7, 0.7831), (69, 0.05), (150, 100.0), (4099, 0.5)])
def test_field_lists_and_tiles(nwater, cutoff, dtype):
    # (E within 2e-6 / 1e-12 a.u. of the oracle's at the same precision, the
    # bounds of the field tests at 128 waters; sums of every molecule of a box
    # are larger, and scale them)
    announce("field nwater=%d cutoff=%g dtype=%s" % (nwater, cutoff, dtype))
    xyz, box, _ = frames(nwater, 1, 4000 + nwater)
    prec = O.F64 if dtype == torch.float64 else O.F32
    cfg = O.config(imodel=1, ispecies=0, imap=0, cutoff=cutoff)
    s = S.eproj_sites(torch.from_numpy(xyz.copy()).to(DEV), torch.from_numpy(box.copy()).to(DEV), cutoff=cutoff,
                      dtype=dtype).cpu().double().numpy()[0]
    e = O.eproj(prec, cfg, xyz[0], box[0])
    tol = 1e-12 if dtype == torch.float64 else 2e-6
    assert np.abs(s[C.SITE_E] - e).max() < tol * max(1.0, np.abs(e).max())
    if cutoff < 0.1:
        assert not e.any() and not s[C.SITE_E].any()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("nwater,ld", [(1, 4), (32, 64), (32, 200), (33, 68), (65, 132), (96, 192)])
def test_hamiltonian_tiles(nwater, ld, dtype):
    announce("hamiltonian nwater=%d ld=%d dtype=%s" % (nwater, ld, dtype))
    xyz, box, _ = frames(nwater, 2, 5000 + nwater)
    prec = O.F64 if dtype == torch.float64 else O.F32
    cfg = O.config(imodel=1, ispecies=0, imap=0, avef=3400.0)
    b = torch.from_numpy(box.copy()).to(DEV)
    s = S.eproj_sites(torch.from_numpy(xyz.copy()).to(DEV), b, dtype=dtype)
    H = S.hamiltonian(s, b, avef=3400.0, ld=ld).cpu().double().numpy()
    n = 2 * nwater
    assert np.all(H[:, :, n:] == 0.0)
    for f in range(2):
        Hf = H[f, :, :n]
        assert np.array_equal(Hf, Hf.T)
        Ho = O.hamiltonian(prec, cfg, xyz[f], box[f], O.eproj(prec, cfg, xyz[f], box[f]))
        # 3e-3 / 1e-9 cm^-1 at |H| ~ 1e3, as the Hamiltonian tests at 128 waters
        assert np.abs(Hf - Ho).max() < (1e-9 if dtype == torch.float64 else 3e-3) * max(1.0, np.abs(Ho).max() / 1e3)
