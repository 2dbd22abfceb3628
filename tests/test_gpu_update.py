"""The tournament LU's look-ahead (a side stream for the rest of each large update) where its streams could get in each
other's way: several threads factoring at once on streams of their own, more of them than the library keeps side
streams, and a captured call. The factors are those of the plain loop, bit for bit."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu

N = 2304                                                   # 36 panels, the first four with a split update


def _plain(dv, Z):
    from mom25d_amd import _lib as L
    was = L.lib().m25x_lu_lookahead()
    L.call('m25x_lu_set_lookahead', 0)
    try:
        F = dv.getrf(Z.clone(), pivot='tournament')
        torch.cuda.synchronize()
    finally:
        L.call('m25x_lu_set_lookahead', was)
    return F


def _matrix(dv, dt, seed):
    g = torch.Generator(dv.device()).manual_seed(seed)
    return torch.randn(N, N, generator=g, device=dv.device(), dtype=torch.complex128).to(dt)


def _same(a, b):
    return torch.equal(a.LU, b.LU) and torch.equal(a.ipiv, b.ipiv) and torch.equal(a.perm, b.perm)


def test_threads_on_their_own_streams(gpu):
    dv = gpu
    Z = [_matrix(dv, (torch.complex64, torch.complex128)[i % 2], i) for i in range(6)]
    want = [_plain(dv, z) for z in Z]
    got = [None] * len(Z)

    def work(i):
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.default_stream())
        with torch.cuda.stream(s):
            got[i] = [dv.getrf(Z[i].clone(), pivot='tournament') for _ in range(2)]
        s.synchronize()

    th = [threading.Thread(target=work, args=(i,)) for i in range(len(Z))]
    [t.start() for t in th]
    [t.join() for t in th]
    for i, F in enumerate(want):
        assert all(_same(F, g) for g in got[i]), i


def test_captured_call(gpu):
    from mom25d_amd import _lib as L
    dv = gpu
    Z = _matrix(dv, torch.complex64, 9)
    want = _plain(dv, Z)
    A, ipiv, perm = Z.clone(), torch.empty_like(want.ipiv), torch.empty_like(want.perm)
    info = torch.zeros(1, dtype=torch.int32, device=dv.device())
    wb = L.lib().m25x_getrf_work_bytes(L.C64, N)
    work = torch.empty(wb, dtype=torch.uint8, device=dv.device())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        L.call('m25x_getrf', L.C64, L.PIVOT_TOURNAMENT, dv.ptr(A), N, N, dv.ptr(ipiv), dv.ptr(perm), dv.ptr(info),
               dv.ptr(work), wb, dv.stream())
    for _ in range(3):
        A.copy_(Z)
        ipiv.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(A, want.LU) and torch.equal(ipiv, want.ipiv) and torch.equal(perm, want.perm)
        assert _same(dv.getrf(Z.clone(), pivot='tournament'), want)     # eager, between the replays
