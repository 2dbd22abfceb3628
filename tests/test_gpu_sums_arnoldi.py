"""The Arnoldi step's sums (m25x_cgs2) where their split changes: every count of columns (a block's threads are 1, 2, 4
or 8 columns wide), basis sizes around the eight vectors read at a time and around one thread an entry of the sum, and
rows past one a thread; against the same formulas in NumPy, and the same bits on a second call.

Tolerance: a dot product of n terms of unit-norm vectors with |w| has an error below n eps |w| in any order of its sum
(20 000 x 1.1e-16 = 2.2e-12), and in practice near sqrt(n) eps; 1e-12 sqrt(n) max|w| covers both."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,nv", [(1, 8, 1), (31, 7, 8), (33, 6, 9), (129, 2, 7), (300, 1, 63), (905, 5, 51), (905, 4, 63),
                                    (16385, 2, 16), (8193, 4, 17), (20000, 3, 2), (4097, 8, 32)])
def test_step_against_numpy(gpu, n, k, nv):
    dv = gpu
    rng = np.random.default_rng(17 * n + k + nv)
    V = rng.standard_normal((nv + 1, n, k)) + 1j * rng.standard_normal((nv + 1, n, k))
    V /= np.linalg.norm(V, axis=1)[:, None, :]
    V[:nv] /= nv                                           # not orthonormal: |I - V V^H| stays below 2
    W = rng.standard_normal((n, k)) + 1j * rng.standard_normal((n, k))
    w = W.copy()
    h = np.zeros((nv + 1, k), complex)
    for _ in range(2):
        d = np.einsum('irc,rc->ic', V[:nv].conj(), w)
        w = w - np.einsum('irc,ic->rc', V[:nv], d)
        h[:nv] += d
    h[nv] = np.linalg.norm(w, axis=0)
    out = []
    for _ in range(2):
        Vd, Wd = torch.from_numpy(V).to(dv.device()), torch.from_numpy(W).to(dv.device())
        hb = torch.zeros((nv + 1, k), dtype=torch.complex128, device=dv.device())
        dv.cgs2(Vd, nv, Wd, hb)
        out.append((hb.cpu().numpy(), Vd.cpu().numpy(), Wd.cpu().numpy()))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    hg, Vg, Wg = out[0]
    tol = 1e-12 * np.sqrt(n) * np.abs(W).max()
    assert np.abs(hg - h).max() <= tol and np.abs(Wg - w).max() <= tol
    assert np.abs(Vg[nv] * h[nv].real - w).max() <= 2 * tol
    assert np.array_equal(Vg[:nv], V[:nv])
