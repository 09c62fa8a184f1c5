"""FP32 site vectors and couplings, every operation rounded once: the squares of
distances, the root and the quotients as the source writes them, evaluated here
with one rounding to FP32 per operation from a wider type."""

import numpy as np
import pytest
import torch

import calcir_amd as C
from calcir_amd import stages as S
from cases import frames
from conftest import announce

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F = np.float32
W = np.longdouble  # holds a product of two FP32 values exactly, a sum to 64 bits


def _fma(a, b, c):
    return (W(a) * W(b) + W(c)).astype(F)


def _square(d):
    return _fma(d[2], d[2], _fma(d[1], d[1], d[0] * d[0]))


def _root(x):
    return np.sqrt(W(x)).astype(F)


def _quotient(a, b):
    return (W(a) / W(b)).astype(F)


def _image(d, L):
    q = _quotient(d, L)
    return d - L * (np.trunc(q) + np.where(np.abs(q - np.trunc(q)) >= 0.5, np.sign(q), F(0))).astype(F)


@pytest.mark.parametrize("nwater,seed", [(2, 1), (31, 2), (64, 3), (66, 4), (128, 15017)])
def test_couplings_round_once_per_operation(nwater, seed):
    announce("coupling rounding nwater=%d seed=%d" % (nwater, seed))
    xyz, box, _ = frames(nwater, 1, seed)
    b = torch.from_numpy(box.copy()).to(DEV)
    sg = S.eproj_sites(torch.from_numpy(xyz.copy()).to(DEV), b, dtype=torch.float32)
    H = S.hamiltonian(sg, b, avef=3400.0).cpu().numpy()[0]
    s = sg.cpu().numpy()[0]
    n, L = 2 * nwater, [F(v) for v in box[0]]
    x = xyz[0].reshape(nwater, 4, 3)
    with np.errstate(all="ignore"):
        # OH unit vectors
        d = [_image(x[:, 1:3, c].reshape(-1) - np.repeat(x[:, 0, c], 2), L[c]) for c in range(3)]
        r = _root(_square(d))
        for c in range(3):
            assert np.array_equal(s[C.SITE_U + c], _quotient(d[c], r))
        # transition-dipole couplings
        u, p = s[C.SITE_U:C.SITE_U + 3], s[C.SITE_R:C.SITE_R + 3]
        d = [_image(p[c][:, None] - p[c][None], L[c]) for c in range(3)]
        r = _root(_square(d))
        inv = _quotient(F(1), r)
        d = [v * inv for v in d]

        def dot(a, e):
            return _fma(a[2], e[2], _fma(a[0], e[0], a[1] * e[1]))

        ui, uj = [v[:, None] + F(0) * d[0] for v in u], [v[None] + F(0) * d[0] for v in u]
        rb = r * F(18.8973)
        g = _quotient(_fma(F(-3), dot(ui, d) * dot(uj, d), dot(ui, uj)), rb * rb * rb)
        t = s[C.SITE_X] * s[C.SITE_MUP]
        ref = g * (t[:, None] * t[None]) * F(2.1947463e5)
    other = np.arange(n)[:, None] // 2 != np.arange(n)[None] // 2
    assert np.array_equal(H[:n, :n][other], ref[other])
