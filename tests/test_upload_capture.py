"""device.upload, whose pinned buffer is given back when the call returns, is refused while the current stream is being
captured: a replay would copy whatever the buffer holds by then. What goes through it (a batch's item tables, a point's
scalars) was refused under capture when these copies were synchronous. On the CPU, with stand-ins for the capture and for
pinned memory."""
import numpy as np
import pytest
import torch

from mom25d_amd import device as dv


@pytest.mark.parametrize('call', [
    lambda: dv.upload(np.arange(3.0)),
    lambda: dv.zgemm_nk_batched([torch.zeros(2, 2, dtype=torch.complex128)], torch.zeros(2, 1, dtype=torch.complex128), [(0, 1)])])
def test_refused_under_capture(monkeypatch, call):
    empty, asked = torch.empty, []
    monkeypatch.setattr(torch, 'empty', lambda *a, pin_memory=False, **k: empty(*a, **k))
    monkeypatch.setattr(dv, 'device', lambda: torch.device('cpu'))
    monkeypatch.setattr(dv, 'stream', lambda: None)
    monkeypatch.setattr(dv.L, 'call', lambda *a: asked.append(a))
    state = [False]
    monkeypatch.setattr(torch.cuda, 'is_current_stream_capturing', lambda: state[0])
    call()
    n, state[0] = len(asked), True
    with pytest.raises(RuntimeError, match='captured'):
        call()
    assert len(asked) == n
