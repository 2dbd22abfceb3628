"""device.cast_rows and the scaled solve hand the library pointers: a scale of another type, length, layout or device, and
tensors that are not on one device with it, are refused before that. On the CPU, with the library a stand-in."""
import pytest
import torch

from mom25d_amd import device as dv


@pytest.fixture
def calls(monkeypatch):
    got = []
    monkeypatch.setattr(dv.L, 'call', lambda *a: got.append(a[0]))
    monkeypatch.setattr(dv, 'stream', lambda: None)
    return got


X = torch.ones(6, 2, dtype=torch.complex128)
R = torch.ones(6, dtype=torch.float64)


def test_what_fits_goes_through(calls):
    dv.cast_rows(X, dv.c64)
    dv.cast_rows(X, dv.c64, R)
    dv.cast_rows(X.conj()[:, :1], dv.c128, R, torch.zeros(6, 5, dtype=dv.c128)[:, 2:3])
    assert calls == ['m25x_cast_rows'] * 3


@pytest.mark.parametrize('scale, out', [
    (R.float(), None), (R[:5], None), (torch.ones(12, dtype=torch.float64)[::2], None), (R[:, None], None),
    (R.to(torch.complex128), None), (R.to('meta'), None),
    (None, torch.zeros(6, 2, dtype=dv.c64)), (None, torch.zeros(5, 2, dtype=dv.c128)), (None, torch.zeros(2, 6, dtype=dv.c128).t()),
    (None, torch.zeros(6, 2, dtype=dv.c128, device='meta'))])
def test_what_does_not_is_refused(calls, scale, out):
    with pytest.raises(ValueError):
        dv.cast_rows(X, dv.c128, scale, out)
    assert not calls
