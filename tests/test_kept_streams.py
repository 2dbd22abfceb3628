"""What the package keeps on the device between calls - a frequency's tables, the near pairs' analytic moments, the parts of
the matrix-free operator - used on another stream than the one that it was queued on: that stream waits for it, and the
allocator is told; on its own stream nothing waits; a call that is being captured waits for nothing outside the capture,
nothing waits for a stream that is being captured, and moments that a capture fills are not taken for filled. A stream
that is not torch's own is not asked for anything later. Streams and the library are stand-ins that note what they are
asked, on the CPU."""
import contextlib
import types

import numpy as np
import pytest
import torch

from mom25d_amd import device as dv


class Stream:
    made = {}

    def __init__(self, stream_id):
        self.made[stream_id] = self
        self.waits, self.cuda_stream, self.stream_id, self.capturing, self.gone = [], id(self), stream_id, False, False
        self.events = 0

    def record_event(self, event=None):
        assert not self.gone and not self.capturing
        self.events += 1
        return ('queued on', self)

    def wait_event(self, e):
        self.waits.append(e)


@pytest.fixture
def cuda(monkeypatch):
    c = types.SimpleNamespace(a=Stream(0), b=Stream(3), calls=[], recorded=[])
    c.now = c.a

    @contextlib.contextmanager
    def on(s):
        was, c.now = c.now, s
        yield
        c.now = was

    monkeypatch.setattr(torch.cuda, 'stream', on)
    monkeypatch.setattr(torch.cuda, 'Stream', lambda stream_id, device_index, device_type: Stream.made[stream_id])
    monkeypatch.setattr(dv, '_current', lambda: (c.now.stream_id, 0, 1), raising=False)
    monkeypatch.setattr(torch.cuda, 'current_stream', lambda device=None: c.now)
    monkeypatch.setattr(torch.cuda, 'is_current_stream_capturing', lambda: c.now.capturing)
    monkeypatch.setattr(torch.Tensor, 'record_stream', lambda t, s: c.recorded.append((t.data_ptr(), s)))
    monkeypatch.setattr(dv, 'device', lambda: torch.device('cpu'))
    monkeypatch.setattr(dv, 'upload', lambda *a: [torch.from_numpy(np.ascontiguousarray(x)) for x in a])
    monkeypatch.setattr(dv.L, 'call', lambda name, *a: c.calls.append((name, a)))
    return c


def _tables(dimg=0.0):
    one = np.ones(1)
    scal = dict(dr=one, d=0 * one, dimg=dimg * one, cA=one, cq=one, cAi=one, cqi=one)
    return dv.DevTables.packed(torch.zeros(1, 4, 4, dtype=torch.float64), scal, np.zeros((1, 1), np.int32), np.zeros(1))


def _plan(n=5):
    z = torch.zeros(n, dtype=torch.int32)
    p = dv.NearPlan.__new__(dv.NearPlan)
    p.P = p.Q = z
    p.n, p.stat, p.stat_ready, p.stat_kind, p.stat_made = n, torch.zeros(n, 12, dtype=torch.float64), False, None, None
    return p


MESH = types.SimpleNamespace(struct=dv.L.Mesh(), quad=dv.L.Quad(), Ne=4, Nt=4)


def _ready(cuda):
    """The stat pointer and the ready flag of the last m25x_near_moments call."""
    a = cuda.calls[-1][1]
    return a[7].value, a[8]


def test_tables(cuda):
    t = _tables()
    assert t.struct.ntab == 1 and not cuda.a.waits and not cuda.recorded          # their own stream: no wait
    cuda.now = cuda.b
    assert t.struct.ntab == 1 and cuda.b.waits == [('queued on', cuda.a)]
    assert {(x.data_ptr(), cuda.b) for x in (t.AQ, t.dr, t.cA, t.tab)} <= set(cuda.recorded)
    assert t.struct.ntab == 1 and cuda.a.events == 1 and len(cuda.b.waits) == 2   # what came later is not waited for
    cuda.b.capturing = True
    assert t.struct.ntab == 1 and len(cuda.b.waits) == 2
    cuda.now, cuda.b.capturing = cuda.a, False
    t = _tables()
    cuda.now, cuda.a.capturing = cuda.b, True
    assert t.struct.ntab == 1 and len(cuda.b.waits) == 2 and cuda.a.events == 1


def test_stream_of_another_library(cuda):
    cuda.now = cuda.a = Stream(stream_id=4096)
    t = _tables()
    cuda.a.gone, cuda.now = True, cuda.b
    assert t.struct.ntab == 1 and cuda.b.waits == [('queued on', cuda.a)]


def test_moments(cuda):
    t, p = _tables(), _plan()
    dv.near_moments(MESH, t, p, 1.0)
    first = _ready(cuda)
    dv.near_moments(MESH, t, p, 1.0)
    assert first == (p.stat.data_ptr(), 0) and _ready(cuda) == (p.stat.data_ptr(), 1) and not cuda.a.waits
    made = cuda.a.events                                                          # once a mesh: recorded at once
    cuda.now = cuda.b
    dv.near_moments(MESH, _tables(), p, 1.0)                                      # tables of its own, the moments kept
    assert made == 1 and cuda.a.events == 1
    assert cuda.b.waits == [('queued on', cuda.a)] and (p.stat.data_ptr(), cuda.b) in cuda.recorded
    assert _ready(cuda) == (p.stat.data_ptr(), 1)
    old = p.stat                                                                  # other parts extracted: filled again,
    dv.near_moments(MESH, _tables(1e-3), p, 1.0)                                  # beside what stream a may still read
    assert _ready(cuda) == (p.stat.data_ptr(), 0) and p.stat.data_ptr() != old.data_ptr()
    cuda.now = cuda.a
    dv.near_moments(MESH, _tables(1e-3), p, 1.0)
    assert cuda.a.waits == [('queued on', cuda.b)]


def test_moments_under_capture(cuda):
    t, p = _tables(), _plan()
    cuda.now.capturing = True
    dv.near_moments(MESH, t, p, 1.0)
    assert _ready(cuda)[1] == 0
    cuda.now.capturing = False
    dv.near_moments(MESH, t, p, 1.0)                                              # the replay may never have come
    assert _ready(cuda)[1] == 0
    cuda.now.capturing = True
    dv.near_moments(MESH, t, p, 1.0)
    assert _ready(cuda)[1] == 1


def test_operator(cuda, monkeypatch):
    """assemble on one stream, matvec_exact on another."""
    from mom25d_amd.fast import FastOperator
    fo = FastOperator.__new__(FastOperator)
    log = types.SimpleNamespace(timer=lambda *a, **k: __import__('contextlib').nullcontext())
    fo.sim = types.SimpleNamespace(Ne=4, Nv=1, log=log)
    fo.mesh, fo.plan = MESH, None
    for name in ('fill_far', 'near_scatter', 'matvec_far', 'csr_matvec', 'via_matvec'):
        monkeypatch.setattr(dv, name, lambda *a, **k: None)
    monkeypatch.setattr(dv, 'near_values', lambda *a: torch.zeros(3, dtype=torch.complex128))
    z = lambda *s: torch.zeros(*s, dtype=torch.complex128)
    lumped = (torch.zeros(1, dtype=torch.int64), torch.zeros(1, dtype=torch.int64), z(1))
    st = dict(f=1.0, w=1.0, tabs=None, M=z(5, 7), B=z(4, 1), C=z(1, 1), lumped=lumped)
    fo.assemble(st, dtype=dv.c64)
    X = z(5, 2)
    fo.matvec_exact(X)
    assert not cuda.a.waits
    cuda.now = cuda.b
    fo.matvec_exact(X)
    assert ('queued on', cuda.a) in cuda.b.waits
    assert {(x.data_ptr(), cuda.b) for x in (st['B'], st['C'], *lumped, fo._op['vals'])} <= set(cuda.recorded)
    fo.assemble(st, dtype=dv.c128)                                                # the values are computed at first use
    cuda.now = cuda.a
    fo.matvec_exact(X)
    cuda.now = cuda.b
    n = len(cuda.b.waits)
    fo.matvec_exact(X)
    assert cuda.a.waits and len(cuda.b.waits) == n + 1 and (fo._op['vals'].data_ptr(), cuda.b) in cuda.recorded
