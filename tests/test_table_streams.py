"""A model's tables are complete when they are kept: a call on another stream reads them
without a wait of its own."""
import types

import numpy as np
import pytest
import torch

from pytransit_amd import RoadRunnerModel, _lib
from pytransit_amd import rrmodel as rrmod

CPU = torch.device('cpu')


@pytest.fixture
def log(monkeypatch):
    """Order of the launches (stood in for) and waits; each wait with the kept tables."""
    events = []
    lib = types.SimpleNamespace(rr_weights_3d=lambda *a: events.append('weights') or 0,
                                rr_ld_basis_count=lambda law: 2,
                                rr_ld_basis_table=lambda *a: events.append('basis') or 0)
    monkeypatch.setattr(_lib, 'load', lambda require_gpu=True: lib)
    monkeypatch.setattr(rrmod, 'stream_handle', lambda device: 0)
    monkeypatch.setattr(_lib, 'synchronize_stream', lambda device: events.append('wait'), raising=False)
    return events


def test_weight_table_is_waited_for_before_it_is_kept(log, monkeypatch):
    m = RoadRunnerModel.__new__(RoadRunnerModel)
    m.klims, m.nk, m.ng, m.ze, m.mu, m.ldname = (0.01, 0.2), 4, 6, np.zeros(5), np.zeros(5), 'quadratic'
    m._tables = {}
    kept = []
    monkeypatch.setattr(_lib, 'synchronize_stream', lambda device: (log.append('wait'), kept.append(dict(m._tables))),
                        raising=False)
    m._table(CPU)
    assert log[:2] == ['weights', 'wait'] and kept[0] == {} and CPU in m._tables
    m._table(CPU)
    assert log.count('weights') == 1


def test_basis_table_is_waited_for(log):
    tab = types.SimpleNamespace(nk=4, ng=6)
    RoadRunnerModel._basis_table(2, _lib.RRTable(nk=tab.nk, ng=tab.ng), CPU)
    assert log == ['basis', 'wait']


def test_the_wait_is_for_the_current_stream(monkeypatch):
    seen = []
    stream = types.SimpleNamespace(synchronize=lambda: seen.append('waited'))
    monkeypatch.setattr(torch.cuda, 'current_stream', lambda device: seen.append(device) or stream)
    dev = torch.device('cuda', 1)
    _lib.synchronize_stream(CPU)
    assert seen == []
    _lib.synchronize_stream(dev)
    assert seen == [dev, 'waited']


@pytest.mark.gpu
@pytest.mark.parametrize('law,nc', [('quadratic', 2), ('nonlinear', 4), ('power-2', 2)])
def test_first_calls_on_two_streams(gpu, law, nc):
    """The first call builds the tables on one stream, the next reads them on another."""
    t = np.linspace(-0.1, 0.1, 500)
    args = (torch.full((3, 1), 0.1, dtype=torch.float64, device=gpu), torch.full((3, 1, nc), 0.2, dtype=torch.float64, device=gpu),
            torch.zeros((3, 1), dtype=torch.float64, device=gpu)) + tuple(
                torch.full((3,), x, dtype=torch.float64, device=gpu) for x in (3.0, 9.0, 1.54, 0.0, 0.0))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(gpu) for _ in range(2)]
    m = RoadRunnerModel(law, device=gpu)
    m.set_data(t)
    out = []
    for s in streams:
        with torch.cuda.stream(s):
            out.append(m.evaluate(*args, copy=False))
    torch.cuda.synchronize()
    ref = m.evaluate(*args)
    assert ref.min() < 0.995
    for f in out:
        assert np.array_equal(f.cpu().numpy(), ref)


def test_only_evaluate_makes_the_basis_table(monkeypatch):
    """lnlike, the weights property, TSModel and the server's model do without; the first
    evaluate makes it once."""
    made = []
    lib = types.SimpleNamespace(rr_weights_3d=lambda *a: 0)
    monkeypatch.setattr(_lib, 'load', lambda require_gpu=True: lib)
    monkeypatch.setattr(rrmod, 'stream_handle', lambda device: 0)
    monkeypatch.setattr(RoadRunnerModel, '_basis_table', staticmethod(lambda law, tab, device: made.append(law) or 'basis'))
    # a device that says it is a GPU, with tensors on the CPU
    class Device:
        type = 'cuda'
    for f in ('as_tensor', 'empty'):
        real = getattr(torch, f)
        monkeypatch.setattr(torch, f, lambda *a, real=real, device=None, **k: real(*a, **k))
    monkeypatch.setattr(_lib, 'synchronize_stream', lambda device: None)
    capturing = []
    monkeypatch.setattr(torch.cuda, 'is_current_stream_capturing', lambda: bool(capturing))
    m = RoadRunnerModel.__new__(RoadRunnerModel)
    m.klims, m.nk, m.ng, m.ze, m.mu, m.ldname = (0.01, 0.2), 4, 6, np.zeros(5), np.zeros(5), 'quadratic'
    m._tables = {}
    dev = Device()
    assert 'basis' not in m._table(dev)[1] and made == []
    capturing.append(True)
    assert 'basis' not in m._table(dev, basis=True)[1] and made == []
    capturing.clear()
    tab = m._table(dev)[0]
    assert m._table(dev, basis=True)[1]['basis'] == 'basis' and m._table(dev, basis=True)[0] is tab and len(made) == 1


@pytest.mark.gpu
def test_first_evaluate_under_capture(gpu):
    """A model whose weight table exists but not its basis table: the captured setup reads the
    weights, and every replay gives the eager flux to rounding (FP64, 1e-12)."""
    t = np.linspace(-0.1, 0.1, 700)
    m, ref = RoadRunnerModel('quadratic', device=gpu), RoadRunnerModel('quadratic', device=gpu)
    for x in (m, ref):
        x.set_data(t, nsamples=3, exptimes=0.01)
    col = lambda *v: torch.as_tensor(v, dtype=torch.float64, device=gpu)
    k, ldc, t0 = col(0.1, 0.05)[:, None], col(0.4, 0.2, 0.3, 0.1).reshape(2, 1, 2), col(0.001, 0.0)[:, None]
    orbit = (col(3.0, 2.5), col(9.0, 8.0), col(1.55, 1.53), col(0.0, 0.1), col(0.0, 0.4))
    m.lnlike(k, ldc, t0, *orbit[:3], np.ones(700), 1e-3)     # uploads the data and makes the weight table
    assert 'basis' not in m._table(gpu)[1]
    stream = torch.cuda.Stream(gpu)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        out = m.evaluate(k, ldc, t0, *orbit, copy=False)
    assert 'basis' not in m._table(gpu)[1]
    for replay in range(3):
        k.copy_(col(0.1 + 0.01 * replay, 0.05)[:, None])
        g.replay()
        torch.cuda.synchronize()
        f = ref.evaluate(k, ldc, t0, *orbit)
        assert f.min() < 0.995 and np.abs(out.cpu().numpy() - f).max() <= 1e-12
    again = m.evaluate(k, ldc, t0, *orbit)
    assert 'basis' in m._table(gpu)[1] and np.array_equal(again, f)
