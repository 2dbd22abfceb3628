"""gmres_batched with operators of every kind that a caller may hand it, on the CPU: the fused step's entry points are
replaced by the formulas that m25x.h states for them (m25x_cgs2_cols changes w, m25x_cgs2_keep does not), reading and
writing through the pointers that the wrapper passes. An operator's result may be its argument or a tensor that its owner
keeps, and of another type; a tensor that the step would misread is refused."""
import ctypes as C

import numpy as np
import pytest
import torch

from mom25d_amd import device as dv
from mom25d_amd.linalg import gmres_batched


def _at(p, shape):
    n = int(np.prod(shape))
    return np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_double)), (2 * n,)).view(complex).reshape(shape)


class _Lib:
    @staticmethod
    def m25x_cgs2_cols_work_bytes(k):
        return 16


@pytest.fixture
def step(monkeypatch):
    def call(name, V, n, k, nv, w, hcol, vnext, work, nbytes, stream):
        assert name in ('m25x_cgs2_cols', 'm25x_cgs2_keep')
        V, w, H, out = _at(V, (nv, n, k)), _at(w, (n, k)), _at(hcol, (nv + 1, k)), _at(vnext, (n, k))
        x = w if name == 'm25x_cgs2_cols' else out
        h1 = np.einsum('irc,rc->ic', V.conj(), w)
        x[...] = w - np.einsum('irc,ic->rc', V, h1)
        h2 = np.einsum('irc,rc->ic', V.conj(), x)
        x[...] = x - np.einsum('irc,ic->rc', V, h2)
        nrm = np.linalg.norm(x, axis=0)
        H[:nv], H[nv] = h1 + h2, nrm
        out[...] = x / np.where(nrm > 0, nrm, 1)

    monkeypatch.setattr(dv.L, 'call', call)
    monkeypatch.setattr(dv.L, 'lib', lambda: _Lib)
    monkeypatch.setattr(dv, 'stream', lambda: None)


N, K = 12, 9                                               # more than eight columns: nothing needs a device


def _system(seed=0):
    g = torch.Generator().manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g, dtype=torch.complex128)
    return torch.eye(N, dtype=torch.complex128) + 0.1 * rnd(N, N), rnd(N, K)


@pytest.mark.parametrize('kind', ['argument', 'kept', 'complex64', 'real', 'conjugate', 'transposed', 'fresh'])
def test_any_operator(step, kind):
    Z, B = _system()
    kept = torch.empty(N, K, dtype=torch.complex128)
    tol = 1e-10
    if kind == 'argument':
        Z, A = torch.eye(N, dtype=torch.complex128), lambda V: V
    elif kind == 'kept':                                   # the result's owner reads it again afterwards
        last = []

        def A(V):
            if last:
                assert torch.equal(kept, last[-1])
            kept.copy_(Z @ V)
            last.append(kept.clone())
            return kept
    elif kind == 'complex64':
        A, tol = (lambda V: (Z @ V).to(torch.complex64)), 1e-5
    elif kind == 'real':                                   # a real operator on real right-hand sides
        Z, B = Z.real.to(torch.complex128), B.real.to(torch.complex128)
        A = lambda V: (Z @ V).real
    elif kind == 'conjugate':
        A = lambda V: (Z.conj() @ V.conj()).conj()
    elif kind == 'transposed':
        A = lambda V: (V.t() @ Z.t()).t()
    else:
        A = lambda V: Z @ V
    X, it = gmres_batched(A, B, rtol=tol, restart=N + 2, maxiter=3)
    assert torch.linalg.vector_norm(Z @ X - B) <= 10 * tol * torch.linalg.vector_norm(B)
    assert kind != 'argument' or it == [1] * K


def test_step_refuses_what_it_would_misread(step):
    V = torch.zeros(4, N, K, dtype=torch.complex128)
    V[0, 0] = 1
    W, h = torch.ones(N, K, dtype=torch.complex128), torch.zeros(4, K, dtype=torch.complex128)
    dv.cgs2(V, 1, W, h)
    bad = [(W.to(torch.complex64), h), (W.real.contiguous(), h), (W.conj(), h), (W.to('meta'), h), (W[:, :K - 1], h),
           (W, h.to(torch.complex64)), (W, h[:1]), (W, h[:, :1].contiguous())]
    for w, hc in bad:
        with pytest.raises(ValueError):
            dv.cgs2(V, 1, w, hc)
