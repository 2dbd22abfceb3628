"""The products' wrappers hand the library a pointer, so an argument whose conjugation torch has put off is conjugated
first, whatever the number of columns: the values at the pointer are the argument's. On the CPU, with the library a stand-in
that reads what it is handed."""
import ctypes as C
import types

import numpy as np
import pytest
import torch

from mom25d_amd import device as dv

N = 6


def _at(p, rows, k, ld):
    p = p.value if hasattr(p, 'value') else p
    n = (rows - 1) * ld + k
    v = np.ctypeslib.as_array(C.cast(C.c_void_p(p), C.POINTER(C.c_double)), (2 * n,)).view(complex)
    return np.stack([v[r * ld:r * ld + k] for r in range(rows)])


@pytest.fixture
def read(monkeypatch):
    got = []

    def call(name, *a):
        if name == 'm25x_matvec_far':
            got.append(_at(a[0], N, a[1], a[2]))
        elif name == 'm25x_csr_matvec':
            got.append(_at(a[4], N, a[5], a[6]))
        elif name == 'm25x_zgemm_nk':
            got.append(_at(a[3], N, a[4], a[4]))
        elif name == 'm25x_zgemm_nk_batched':
            got.extend(_at(it.X, N, it.k, it.ldx) for it in a[1])
        elif name == 'm25x_via_matvec':
            got.extend([_at(a[4], N, a[5], a[6]), _at(a[0], N - 1, 1, 1), _at(a[1], 1, 1, 1)])

    monkeypatch.setattr(dv.L, 'call', call)
    monkeypatch.setattr(dv.L, 'lib', lambda: types.SimpleNamespace(m25x_matvec_far_work_bytes=lambda *a: 16,
                                                                   m25x_via_matvec_work_bytes=lambda *a: 16))
    monkeypatch.setattr(dv, 'stream', lambda: None)
    monkeypatch.setattr(dv, '_call_table', lambda cls, its: (its, torch.zeros(1)))
    return got


MESH = types.SimpleNamespace(struct=dv.L.Mesh(), Ne=N, Nt=4)
TABS = types.SimpleNamespace(struct=dv.L.Tables())
PLAN = types.SimpleNamespace(rowptr=torch.zeros(N + 1, dtype=torch.int32), ecol=torch.zeros(1, dtype=torch.int32))
Z = torch.zeros(N, N, dtype=torch.complex128)


def _via(X):
    B = torch.arange(1, N, dtype=torch.float64) * (1 + 1j)
    dv.via_matvec(B[:, None].conj(), torch.full((1, 1), 2j).to(torch.complex128).conj(), X, torch.zeros_like(X))


@pytest.mark.parametrize('k', [1, 8, 9, 20])
@pytest.mark.parametrize('call', [
    lambda X: dv.matvec_far(X, MESH, TABS, 1.0),
    lambda X: dv.csr_matvec(PLAN, torch.zeros(1), X),
    lambda X: dv.zgemm_nk(Z, X),
    lambda X: dv.zgemm_nk_batched([Z], X, [(0, X.shape[1])]),
    _via])
def test_values_at_the_pointer(read, call, k):
    X = torch.randn(N, k, dtype=torch.complex128, generator=torch.Generator().manual_seed(k))
    for arg in (X, X.conj(), X.to(torch.complex64).conj(), X.t().conj().contiguous().t()):
        if call is _via and not (arg.dtype == torch.complex128 and arg.is_contiguous()):
            continue                                       # (refused)
        read.clear()
        call(arg)
        want = arg.resolve_conj().to(torch.complex128).numpy()
        if call is _via:
            assert np.array_equal(read[0], want) and np.array_equal(read[1][:, 0], np.arange(1, N) * (1 - 1j))
            assert read[2][0, 0] == -2j
        else:
            assert np.array_equal(np.concatenate(read, axis=1), want)
