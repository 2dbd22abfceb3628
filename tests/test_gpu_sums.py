"""The matrix-free operator's via part and its sparse near part against plain products in complex128."""
import types

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _cx(rng, *shape):
    return torch.from_numpy(rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).cuda()


@pytest.mark.parametrize('ne,nv,k', [(1, 1, 1), (5, 3, 4), (31, 2, 5), (257, 10, 8), (1000, 1, 9), (8200, 40, 3)])
def test_via_matvec(ne, nv, k):
    """Sums of up to 8200 products: within 1e-12 of each row's absolute sum (8200 x 2^-53 = 9e-13)."""
    from mom25d_amd import device as dv
    rng = np.random.default_rng(ne + nv + k)
    B, C, X, Y0 = _cx(rng, ne, nv), _cx(rng, nv, nv), _cx(rng, ne + nv, k), _cx(rng, ne + nv, k)
    Y = Y0.clone()
    dv.via_matvec(B, C, X, Y)
    b, c, x, y = (t.cpu().numpy() for t in (B, C, X, Y0))
    want = np.concatenate([y[:ne] + b @ x[ne:], b.T @ x[:ne] + c @ x[ne:]])
    size = np.concatenate([abs(y[:ne]) + abs(b) @ abs(x[ne:]), abs(b.T) @ abs(x[:ne]) + abs(c) @ abs(x[ne:])])
    assert (np.abs(Y.cpu().numpy() - want) <= 1e-12 * size).all()


@pytest.mark.parametrize('k', [1, 3, 8, 11])
@pytest.mark.parametrize('add', [False, True])
def test_csr_matvec(k, add):
    """Rows of 0, 1, 63, 64, 65 and 300 entries (sums of 300 products: within 1e-13 of the absolute sum)."""
    from mom25d_amd import device as dv
    rng = np.random.default_rng(k)
    lens = [0, 1, 63, 64, 65, 300, 0, 2]
    n = 400
    rowptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(n, m, replace=False)) for m in lens]).astype(np.int32)
    plan = types.SimpleNamespace(rowptr=torch.from_numpy(rowptr).cuda(), ecol=torch.from_numpy(col).cuda())
    v, X, Y0 = _cx(rng, len(col)), _cx(rng, n, k), _cx(rng, len(lens), k)
    got = dv.csr_matvec(plan, v, X, Y0.clone() if add else None).cpu().numpy()
    A = np.zeros((len(lens), n), complex)
    for r in range(len(lens)):
        A[r, col[rowptr[r]:rowptr[r + 1]]] = v.cpu().numpy()[rowptr[r]:rowptr[r + 1]]
    x, y = X.cpu().numpy(), Y0.cpu().numpy() * add
    assert (np.abs(got - (y + A @ x)) <= 1e-13 * (abs(y) + abs(A) @ abs(x)) + 1e-300).all()
