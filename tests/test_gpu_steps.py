"""gmres_batched on the device with operators whose results are not the step's to change, or not of its type: the argument
itself, a tensor that its owner keeps, complex64, real, a lazy conjugate; below and above eight columns. And the step that
keeps w: the bits of the one that overwrites it, w as it was.

Tolerance: the solves run to a residual of rtol |b| by their own estimate, which the true residual meets within a factor
that a well-conditioned system of this size keeps well below 10 (complex64 results: eps32 = 6e-8 a product, rtol 1e-5)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('k', [3, 8, 9, 20])
@pytest.mark.parametrize('kind', ['argument', 'kept', 'complex64', 'real', 'conjugate', 'transposed'])
def test_any_operator(gpu, kind, k):
    from mom25d_amd.linalg import gmres_batched
    n, rtol = 300, 1e-10
    print(f"operators: {kind} k={k}", flush=True)
    g = torch.Generator(gpu.device()).manual_seed(k)
    rnd = lambda *s: torch.randn(*s, generator=g, dtype=torch.complex128, device=gpu.device())
    Z, B = torch.eye(n, dtype=torch.complex128, device=gpu.device()) + 0.02 * rnd(n, n), rnd(n, k)
    kept, was, same = {}, {}, []                           # a kept result for each count of columns, and its values
    if kind == 'argument':
        Z, A = torch.eye(n, dtype=torch.complex128, device=gpu.device()), lambda V: V
    elif kind == 'kept':
        def A(V):
            c = V.shape[1]
            if c in was:
                same.append((kept[c] == was[c]).all())
            kept[c] = kept.get(c, torch.empty_like(V)).copy_(Z @ V)
            was[c] = kept[c].clone()
            return kept[c]
    elif kind == 'complex64':
        A, rtol = (lambda V: (Z @ V).to(torch.complex64)), 1e-5
    elif kind == 'real':
        Z, B = Z.real.to(torch.complex128), B.real.to(torch.complex128)
        A = lambda V: (Z @ V).real
    elif kind == 'conjugate':
        A = lambda V: (Z.conj() @ V.conj()).conj()
    else:
        A = lambda V: (V.t().contiguous() @ Z.t().contiguous()).t()
    X, it = gmres_batched(A, B, rtol=rtol, restart=40, maxiter=3)
    assert (torch.linalg.vector_norm(Z @ X - B, dim=0) <= 10 * rtol * torch.linalg.vector_norm(B, dim=0)).all()
    if kind == 'kept':
        assert len(same) > 3 and all(bool(s) for s in same)


@pytest.mark.parametrize('n,k,nv', [(1, 1, 1), (33, 6, 9), (905, 4, 63), (4097, 8, 17), (513, 130, 2)])
def test_step_that_keeps_w(gpu, n, k, nv):
    dv = gpu
    g = torch.Generator(dv.device()).manual_seed(n + k + nv)
    V = torch.randn(nv + 1, n, k, generator=g, dtype=torch.complex128, device=dv.device())
    V /= torch.linalg.vector_norm(V, dim=1)[:, None, :]
    V[:nv] /= nv
    W = torch.randn(n, k, generator=g, dtype=torch.complex128, device=dv.device())
    h = [torch.zeros(nv + 1, k, dtype=torch.complex128, device=dv.device()) for _ in range(2)]
    Va, Wa, Vb, Wb = V.clone(), W.clone(), V.clone(), W.clone()
    dv.cgs2(Va, nv, Wa, h[0])
    dv.cgs2(Vb, nv, Wb, h[1], keep=True)
    assert torch.equal(Va, Vb) and torch.equal(h[0], h[1]) and torch.equal(Wb, W) and torch.equal(Va[:nv], V[:nv])
