"""A batch's solve of more than eight columns of one factor goes in parts of eight, all in one launch: each part has a
workspace of its own (the parts run at once). The item table that the wrapper builds is looked at on the CPU; the library
is a stand-in."""
import types

import pytest
import torch

from mom25d_amd import device as dv

BYTES = 4096


@pytest.fixture
def items(monkeypatch):
    got = []
    monkeypatch.setattr(dv, 'device', lambda: torch.device('cpu'))
    monkeypatch.setattr(dv.L, 'lib', lambda: types.SimpleNamespace(m25x_getrs_work_bytes=lambda code, n, ldb: BYTES))
    monkeypatch.setattr(dv.L, 'call', lambda *a: None)
    monkeypatch.setattr(dv, 'stream', lambda: None)
    monkeypatch.setattr(dv, 'cast_rows', lambda R, dtype: R.to(dtype))
    monkeypatch.setattr(dv, '_call_table', lambda cls, its: (got.extend(its), torch.zeros(1))[1:] * 2)
    monkeypatch.setattr(dv, '_solve_fault', lambda d: torch.zeros(1, dtype=torch.int32))
    return got


@pytest.mark.parametrize('ks', [(8, 3), (9, 2), (20, 8, 17)])
def test_parts_have_workspaces_of_their_own(items, ks):
    n = 6
    F = [dv.Factor(torch.zeros(n, n, dtype=torch.complex64), *(torch.zeros(n, dtype=torch.int32) for _ in range(3))) for _ in ks]
    first = [sum(ks[:i]) for i in range(len(ks))]
    solve = dv.BatchSolve(F, list(zip(first, ks)))
    for subset in (None, [(c, min(k, 10)) for c, k in zip(first, ks)]):
        items.clear()
        solve(torch.zeros(n, sum(ks), dtype=torch.complex128), subset=subset)
        want = ks if subset is None else [min(k, 10) for k in ks]
        assert sum(it.nrhs for it in items) == sum(want) and len(items) == sum(-(-k // 8) for k in want)
        at = sorted(it.work for it in items)
        assert all(b - a >= BYTES for a, b in zip(at, at[1:])) and all(it.work_bytes >= BYTES for it in items)
