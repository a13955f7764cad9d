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
