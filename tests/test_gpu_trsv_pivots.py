"""The complex64 solves, whose diagonal blocks are FP64 inverses, on factors with small pivots: rows graded over seven
decades, and three pivots of 2e-4 in one 64-row block and three in the block before it (blocks' conditions, asserted, up to
the 5e8 at which an FP64 inverse is as exact as FP32 substitution), past the first blocks of a chain in either order; with a
row permutation. The backward error of substitution, row by row, as an FP64 evaluation of the two products gives it.

Tolerance, that of a substitution in FP32: 3 n eps |L| |U| |x|, times 2 sqrt(2) for complex products, and one rounding each
of b and x."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


def _block_condition(U, b):
    T = U[64 * b:64 * b + 64, 64 * b:64 * b + 64]
    return np.abs(np.abs(np.linalg.inv(T)) @ np.abs(T)).sum(1).max()


@pytest.mark.parametrize('kind', ['graded rows', 'graded columns', 'small pivots'])
@pytest.mark.parametrize('n', [1100, 1152])                # 18 blocks, the last one ragged or whole
def test_backward_error(gpu, kind, n):
    dv = gpu
    rng = np.random.default_rng(n)
    cplx = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)
    lu = 0.02 * cplx(n, n)
    lu[np.diag_indices(n)] = np.exp(2j * np.pi * rng.random(n))
    scale = 10.0 ** (-7 * rng.random(n))
    upper = np.triu(np.ones((n, n), bool))
    if kind == 'graded rows':
        lu = np.where(upper, scale[:, None] * lu, lu)
    elif kind == 'graded columns':
        lu = np.where(upper, scale[None, :] * lu, lu)
    else:
        for b in (8, 9):                                   # blocks 8 and 9 of 18, from either end
            for i in (64 * b + 5, 64 * b + 30, 64 * b + 50):
                lu[i, i] *= 2e-4
    lu = lu.astype(np.complex64)
    U, L = np.triu(lu).astype(complex), np.tril(lu, -1) + np.eye(n, dtype=complex)
    if kind == 'small pivots':
        assert all(1e6 <= _block_condition(U, b) <= 5e8 for b in (8, 9))
    perm = rng.permutation(n)
    d = dv.device()
    ints = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).to(d)
    F = dv.Factor(torch.from_numpy(np.ascontiguousarray(lu.T)).to(d), ints(np.arange(n)), ints(perm), ints([0]))
    for k in (1, 4, 7):
        b = cplx(n, k).astype(np.complex64)
        for trans in (0, 1):
            x = dv.getrs(F, torch.from_numpy(b).to(d), trans=trans).cpu().numpy()
            (M0, M1), z, rhs = ((U.T, L.T), x[perm], b) if trans else ((L, U), x, b[perm])
            r = np.abs(M0 @ (M1 @ z) - rhs)
            bound = np.abs(M0) @ (np.abs(M1) @ np.abs(z))
            assert np.all(r <= 3 * n * 2 * np.sqrt(2) * EPS * bound + 2 * EPS * np.abs(rhs)), (k, trans)
    assert not dv.solve_faults()
