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
                                    (16385, 2, 16), (8193, 4, 17), (20000, 3, 2), (4097, 8, 32),
                                    (700, 9, 3), (1100, 16, 8), (905, 24, 33), (300, 67, 6), (513, 130, 2), (5, 1025, 4)])
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


@pytest.mark.parametrize("dst", [torch.complex64, torch.complex128])
@pytest.mark.parametrize("form", ["c128", "c64", "columns", "transposed", "conj", "real", "repeated", "one row"])
@pytest.mark.parametrize("scaled", [False, True])
def test_cast_rows_is_product_and_conversion(gpu, form, dst, scaled):
    """Bit for bit the product and the conversion that it stands for, whatever the source's type and strides."""
    dv = gpu
    torch.manual_seed(3)
    dev = dv.device()
    full = torch.randn(333, 9, dtype=torch.complex128, device=dev)
    src = dict(c128=full, c64=full.to(torch.complex64), columns=full[:, 2:5], transposed=full.t(), conj=full.conj()[:, 1:],
               real=full.real, repeated=full[5:6].expand(40, 9))
    src['one row'] = full[7:8, 3:]
    src = src[form]
    r = torch.rand(src.shape[0], dtype=torch.float64, device=dev) + 0.5 if scaled else None
    want = ((src.to(torch.complex128) if r is None else r[:, None] * src.to(torch.complex128)).to(dst)).contiguous()
    keep = src.clone()
    wide = torch.zeros((src.shape[0], src.shape[1] + 3), dtype=dst, device=dev)
    got = dv.cast_rows(src, dst, r)
    dv.cast_rows(src, dst, r, wide[:, 2:2 + src.shape[1]])
    assert got.dtype == dst and torch.equal(got, want) and torch.equal(wide[:, 2:-1], want)
    assert not wide[:, :2].any() and not wide[:, -1:].any() and torch.equal(src, keep)


@pytest.mark.parametrize("k", [1, 4, 11])
@pytest.mark.parametrize("dtype", [torch.complex64, torch.complex128])
def test_scaled_solve(gpu, k, dtype):
    """diag(r) solve(diag(r) B) in one call: the same bits as the two products around the solve."""
    dv = gpu
    torch.manual_seed(4)
    n = 200
    Z = (torch.randn(n, n, dtype=torch.complex128, device=dv.device()) + 30 * torch.eye(n, device=dv.device())).to(dtype)
    F = dv.getrf(Z)
    B = torch.randn(n, k, dtype=torch.complex128, device=dv.device())
    r = torch.rand(n, dtype=torch.float64, device=dv.device()) + 0.5
    assert torch.equal(dv.getrs(F, B, scale=r), r[:, None] * dv.getrs(F, r[:, None] * B))
    assert not dv.solve_faults()


def test_cast_rows_refuses(gpu):
    from mom25d_amd import _lib as L
    t = gpu.ptr(torch.zeros(8, dtype=torch.complex128, device=gpu.device()))
    for bad in [(7, t, 2, 1, t, 2, 2, 2), (L.C128, t, 1, L.C64, t, 2, 2, 2), (L.C128, t, 2, L.C64, t, 1, 2, 2),
                (L.C128, None, 2, L.C64, t, 2, 2, 2), (L.C128, t, 2, L.C64, t, 2, -1, 2)]:
        with pytest.raises(Exception):
            L.call('m25x_cast_rows', *bad, None, gpu.stream())
