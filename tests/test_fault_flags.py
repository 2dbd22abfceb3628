"""The flag that a solve raises when a wait between its workgroups ran out: each stream has one of its own (read, or'ed and
written by kernels of that stream alone, so none is lost between streams), and solve_faults reports those of every stream
of the device, once. On the CPU, the current stream a stand-in."""
import pytest
import torch

from mom25d_amd import device as dv


@pytest.fixture
def on(monkeypatch):
    now = [0]
    monkeypatch.setattr(dv, '_FAULTS', {})
    monkeypatch.setattr(dv, '_current', lambda: (now[0], 0, 1))
    monkeypatch.setattr(torch.cuda, 'is_current_stream_capturing', lambda: now[0] == 'captured')
    return lambda s: now.__setitem__(0, s)


def test_flags_of_two_streams(on):
    d = torch.device('cpu')
    a = dv._solve_fault(d)
    on(3)
    b = dv._solve_fault(d)
    assert a.data_ptr() != b.data_ptr() and dv._solve_fault(d) is b
    assert not dv.solve_faults(d)
    b.bitwise_or_(torch.ones(1, dtype=torch.int32))
    on(0)
    assert dv._solve_fault(d) is a and dv.solve_faults(d) and not dv.solve_faults(d)
    a.fill_(1), b.fill_(1)
    assert dv.solve_faults(d) and not dv.solve_faults(d)
    assert not dv.solve_faults('meta')
    on('captured')                                         # a capture makes none where there is one
    assert dv._solve_fault(d) is a and len(dv._FAULTS) == 2
