"""The tournament's GEPP at its edges: row counts around a sub-panel (8), a panel (64) and a leaf (256), columns of
zeros, and columns whose largest magnitude several rows share (the earliest position wins), against the oracle's pivots."""
import numpy as np
import pytest
import torch

from oracle import lu as olu

pytestmark = pytest.mark.gpu


def _first_panel(A, dtype):
    from mom25d_amd import device as dv
    n = A.shape[0]
    F = dv.getrf(torch.from_numpy(np.ascontiguousarray(A.T)).cuda().to(dtype))
    win = olu.tslu_winners(A, 0, min(64, n), 256, 4)
    return F.ipiv.cpu().numpy()[:len(win)], olu.interchanges(win, 0, np.arange(n))


@pytest.mark.parametrize('n', [1, 7, 8, 9, 63, 64, 65, 71, 255, 256, 257, 1025])
def test_pivots_at_the_edges(n):
    """Random rows (complex128): the oracle's interchanges."""
    rng = np.random.default_rng(n)
    got, want = _first_panel(rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n)), torch.complex128)
    assert np.array_equal(got, want)


@pytest.mark.parametrize('dtype', [torch.complex64, torch.complex128])
@pytest.mark.parametrize('n', [64, 200, 256, 320])
def test_ties_go_to_the_earliest_position(n, dtype):
    """Each row holds one entry of the panel, a unit (1, -1, j or -j), in a column drawn at random: every column's
    rows tie, some columns have none (all zero), and the elimination is exact in either type."""
    rng = np.random.default_rng(n)
    A = np.zeros((n, n), complex)
    A[np.arange(n), rng.integers(0, 64, n)] = 1j ** rng.integers(0, 4, n)
    got, want = _first_panel(A, dtype)
    assert np.array_equal(got, want)
