"""Solves that share the device. A solve's workgroups note which blocks of a chain have started and which are taken, and
wait for no block that neither holds: after a call every block of both triangles has started and was taken, once each, and
nothing past them; calls on several streams and threads at once, each alone larger than the chip, give the bits that they
give one after the other."""
import threading

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _factor(dv, n, dt, seed):
    g = torch.Generator(dv.device()).manual_seed(seed)
    Z = torch.randn(n, n, generator=g, dtype=torch.complex128, device=dv.device())
    Z += n ** 0.5 * torch.eye(n, device=dv.device())
    return dv.getrf(Z.to(dt))


@pytest.mark.parametrize('dt', [torch.complex64, torch.complex128])
@pytest.mark.parametrize('n,k', [(1, 1), (64, 3), (65, 8), (2047, 2), (2049, 7), (4200, 8)])
def test_every_block_is_taken_once(gpu, n, k, dt):
    from mom25d_amd import _lib as L
    dv = gpu
    F = _factor(dv, n, dt, n)
    code, es = (L.C128, 16) if dt == torch.complex128 else (L.C64, 8)
    nb, chains = -(-n // 64), -(-k // 2)
    W = -(-2 * nb // 64)
    wb = L.lib().m25x_getrs_work_bytes(code, n, k)
    for trans in (0, 1):
        B = torch.ones(n, k, dtype=dt, device=dv.device())
        work = torch.zeros(wb, dtype=torch.uint8, device=dv.device())
        L.call('m25x_getrs', code, dv.ptr(F.LU), n, F.LU.stride(0), dv.ptr(F.ipiv), dv.ptr(F.perm), dv.ptr(B), k, k, trans,
               dv.ptr(work), wb, dv.stream())
        room = work[2 * 8 * n * es:3 * 8 * n * es + n * es].cpu().numpy()      # between the solutions and the permutation
        words, rest = room[:8 * 2 * W * chains].view(np.uint64).reshape(chains, 2, W), room[8 * 2 * W * chains:]
        bits = np.unpackbits(words.view(np.uint8), axis=-1, bitorder='little')
        assert bits[:, :, :2 * nb].all() and not bits[:, :, 2 * nb:].any() and not rest.any()


def test_streams_and_threads_at_once(gpu):
    dv = gpu
    n, k, dts = 5000, 8, (torch.complex64, torch.complex128)
    F = [_factor(dv, n, dts[i % 2], i) for i in range(4)]
    B = [torch.randn(n, k, dtype=torch.complex128, device=dv.device()) for _ in F]
    want = [dv.getrs(f, b) for f, b in zip(F, B)]
    torch.cuda.synchronize()
    got = [None] * len(F)

    def work(i):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            got[i] = [dv.getrs(F[i], B[i]) for _ in range(5)]
        s.synchronize()

    th = [threading.Thread(target=work, args=(i,)) for i in range(len(F))]
    [t.start() for t in th]
    [t.join() for t in th]
    assert not dv.solve_faults()
    for w, g in zip(want, got):
        assert all(torch.equal(w, x) for x in g)
