"""The triangular solves on factors with small pivots, at sizes around the first blocks of a chain (which take the tile
before theirs as any other) and the blocks after them (which fold it into their own inverse): the backward error of
substitution, |L U x - b| <= 3 n eps |L| |U| |x| row by row, in both orders and element types."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dt', [np.complex64, np.complex128])
@pytest.mark.parametrize('n', [65, 448, 449, 512, 577, 701])
def test_small_pivots_keep_the_backward_error_of_substitution(gpu, n, dt):
    from mom25d_amd import device as dv
    rng = np.random.default_rng(n)
    cplx = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)
    lu = 0.05 * cplx(n, n)
    lu[np.diag_indices(n)] = np.exp(2j * np.pi * rng.random(n))
    for i in rng.choice(n, 3, replace=False):              # three pivots of 1e-4: a block's condition to about 1e5
        lu[i, i] *= 1e-4
    lu = lu.astype(dt)
    d = dv.device()
    idx = torch.arange(n, dtype=torch.int32, device=d)
    F = dv.Factor(torch.from_numpy(np.ascontiguousarray(lu.T)).to(d), idx, idx, torch.zeros(1, dtype=torch.int32, device=d))
    lu = lu.astype(complex)
    L, U = np.tril(lu, -1) + np.eye(n), np.triu(lu)
    eps = np.finfo(dt).eps / 2
    for k in (1, 2, 7):
        b = cplx(n, k).astype(dt)
        for trans in (0, 1):
            x = dv.getrs(F, torch.from_numpy(b).to(d), trans=trans).cpu().numpy()
            M = (U.T, L.T) if trans else (L, U)            # the product that x solves, first triangle first
            r = np.abs(M[0] @ (M[1] @ x) - b)
            bound = np.abs(M[0]) @ (np.abs(M[1]) @ np.abs(x))
            # complex products: a factor of 2 sqrt(2) on the real bound; b and x are rounded once each
            assert np.all(r <= 3 * n * 2 * np.sqrt(2) * eps * bound + 2 * eps * np.abs(b)), (n, k, trans)
    assert not dv.solve_faults()
