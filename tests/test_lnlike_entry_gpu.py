"""rr_lnlike, the likelihood entry without a workspace (one kernel, the setup in the block),
through the C ABI: against the FP64 oracle with the bars of the likelihood tests, and
against rr_lnlike_vec, whose sums differ in their order only.  Mixed precision sums FP32
sample terms, so the two entries may differ by the mixed bar of 1 ppm a point."""
import ctypes
import math

import numpy as np
import pytest
import torch

from pytransit_amd import RoadRunnerModel, _lib, workloads

pytestmark = pytest.mark.gpu

SIGMA = 300e-6


def entry(model, gpu, k, ldc, t0, p, a, i, obs, grad):
    """lnl and gradient from rr_lnlike; t0 [npv, ncols]."""
    lib = _lib.load()
    npv = len(k)
    dev = lambda x: torch.as_tensor(np.ascontiguousarray(x, dtype=np.float64), device=gpu)
    k, ldc, t0, p, a, i, obs, zero, sig = (dev(x) for x in (k, ldc, t0, p, a, i, obs, np.zeros(npv), np.full(npv, SIGMA)))
    lnl = torch.full((npv + 1,), -7.0, dtype=torch.float64, device=gpu)
    g = torch.full((npv * 7 + 1,), -7.0, dtype=torch.float64, device=gpu) if grad else None
    tab, _keep = model._table(gpu)
    lc = model._lc_descriptor(gpu, 1, t0.shape[1])
    prm = _lib.RRParams(npv, 1, t0.shape[1], 0, *(x.data_ptr() for x in (k, t0, p, a, i, zero, zero)))
    ld = _lib.RRLd(_lib.LD_LAW_IDS[model.ldname][0], ldc.shape[-1], ldc.data_ptr(), 0, 0)
    ref = ctypes.byref
    _lib.check(lib.rr_lnlike(_lib.RR_FP64 if model.precision == 'fp64' else _lib.RR_MIXED, ref(tab), ref(lc), ref(prm), ref(ld),
                             obs.data_ptr(), sig.data_ptr(), lnl.data_ptr(), _lib.ptr(g), _lib.stream_handle(gpu)))
    torch.cuda.synchronize()
    assert lnl[-1].item() == -7.0 and (g is None or g[-1].item() == -7.0)
    return lnl[:-1].cpu().numpy(), None if g is None else g[:-1].reshape(npv, 7).cpu().numpy()


# one time, odd numbers of times and g, several rounds of the queue, unsorted times; epochs in the
# second column; the largest grids that the entry takes (82 KB of LDS with the gradient in FP64)
@pytest.mark.parametrize('npv,npt,nss,law,ng,nz,shuffle', [
    (3, 1, 1, 'quadratic', 100, 40, False), (5, 257, 3, 'power-2', 100, 40, False), (4, 3001, 5, 'quadratic', 51, 40, False),
    (3, 5000, 12, 'power-2', 100, 40, True), (40, 900, 2, 'quadratic', 100, 40, False), (2, 700, 2, 'quadratic', 512, 1024, False)])
@pytest.mark.parametrize('precision', ['fp64', 'mixed'])
def test_rr_lnlike(gpu, oracle, npv, npt, nss, law, ng, nz, shuffle, precision):
    rng = np.random.default_rng(npv + npt)
    pop = workloads.rr_gradient(npv=npv, npt=4, seed=npt).pop
    ldc = np.stack([pop['u1'], pop['u2']], 1) if law == 'quadratic' else rng.uniform(0.4, 0.8, (npv, 2))
    ldc = ldc[:, None, :]
    t = np.linspace(-0.2, 0.2, npt) if npt > 1 else np.array([0.001])
    t = rng.permutation(t) if shuffle else t
    exp = 0.01 if nss > 1 else 0.0
    grid = dict(ng=ng, nzin=nz // 2, nzlimb=nz // 2, nk=8, klims=(0.02, 0.25))   # holds the workload's radius ratios: others give NaN
    m = RoadRunnerModel(law, precision=precision, **grid)
    m.set_data(t, nsamples=nss, exptimes=exp, epids=[1])
    om = oracle.OracleRR(law, **grid)
    om.set_data(t, nsamples=nss, exptimes=exp)
    k, t0, p, a, i = (pop[n] for n in ('k', 't0', 'p', 'a', 'i'))
    f = np.atleast_2d(om.evaluate(k[:, None], ldc, t0[:, None], p, a, i)).reshape(npv, npt)
    obs = f[0] + rng.normal(0, SIGMA, npt)
    r = (obs[None] - f) / SIGMA
    lnl = (-math.log(SIGMA) - 0.5 * math.log(2 * math.pi) - 0.5 * r ** 2).sum(1)
    ppm = 1e-6 * np.abs(r).sum(1) / SIGMA
    bar = 1e-12 * np.abs(lnl) if precision == 'fp64' else ppm
    two = np.column_stack([np.full(npv, 5.0), t0])      # the light curve's epoch is column 1
    got, g = entry(m, gpu, k, ldc, two, p, a, i, obs, True)
    plain, _ = entry(m, gpu, k, ldc, two, p, a, i, obs, False)
    assert (np.abs(got - lnl) <= bar).all() and (np.abs(plain - lnl) <= bar).all()
    vec, gv = m.lnlike(k, ldc, two, p, a, i, obs, SIGMA, grad=True)
    scale = np.abs(gv).max(0)
    assert np.isfinite(gv).all() and (scale > 0).all() or npt == 1
    assert (np.abs(got - vec) <= 2 * bar).all()
    # FP64: the same terms in both entries but for fused steps, each to a few roundings; 1e-9
    # of the largest component allows the sums to cancel a million times.  Mixed: the suite's
    # bar for its gradient, 1e-4 of a component and of its parameter's RMS.
    if precision == 'fp64':
        assert (np.abs(g - gv) <= 1e-9 * scale).all()
    else:
        assert (np.abs(g - gv) <= 1e-4 * (np.abs(gv) + np.sqrt((gv ** 2).mean(0)))).all()


def test_rr_lnlike_invalid_vectors(gpu):
    m = RoadRunnerModel('quadratic')
    m.set_data(np.linspace(-0.1, 0.1, 300))
    one = np.ones(4)
    a = np.array([9.0, 0.8, 9.0, np.nan])
    got, g = entry(m, gpu, np.array([0.1, 0.1, 0.7, 0.1]), np.tile([[0.4, 0.2]], (4, 1, 1)), 0 * one[:, None], 3 * one, a, 1.55 * one,
                   np.ones(300), True)
    assert np.isfinite(got[0]) and np.isfinite(g[0]).all() and np.isnan(got[1:]).all() and np.isnan(g[1:]).all()
