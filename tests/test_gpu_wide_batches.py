"""Batched solves with more than eight columns of one factor in a call (parts of eight side by side), bit for bit the
one-factor solves, which take the parts one after the other."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dt', [torch.complex64, torch.complex128])
@pytest.mark.parametrize('trans', [0, 1])
def test_wide_items(gpu, dt, trans):
    dv = gpu
    ns, ks = (700, 450, 130), (20, 9, 3)
    g = torch.Generator(dv.device()).manual_seed(5)
    rnd = lambda *s: torch.randn(*s, generator=g, dtype=torch.complex128, device=dv.device())
    F = [dv.getrf((rnd(n, n) + n ** 0.5 * torch.eye(n, device=dv.device())).to(dt)) for n in ns]
    R = rnd(max(ns), sum(ks))
    first = [sum(ks[:i]) for i in range(len(ks))]
    solve = dv.BatchSolve(F, list(zip(first, ks)))
    for _ in range(3):
        X = solve(R, trans=trans)
        for f, n, c, k in zip(F, ns, first, ks):
            assert torch.equal(X[:n, c:c + k], dv.getrs(f, R[:n, c:c + k], trans=trans)), n
    assert not dv.solve_faults()
