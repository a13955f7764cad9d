"""The likelihood kernels at the edges of their tiles, queue and splits, and the inputs
they read in place, against the FP64 oracle.  The FP64 sums agree with the oracle's to
a few roundings of the largest term (rtol 1e-12, the suite's bar for lnL).  The mixed
flux has the suite's bar of 1 ppm a point, which moves lnL by at most
1e-6 sum |o - m| / sigma^2."""
import math

import numpy as np
import pytest
import torch

from pytransit_amd import RoadRunnerModel, workloads

pytestmark = pytest.mark.gpu

SIGMA = 300e-6


def make(oracle, npv, npt, nss, law, seed, shuffle=False, span=0.4):
    rng = np.random.default_rng(seed)
    wl = workloads.rr_gradient(npv=npv, npt=4, seed=seed)
    t = np.linspace(-0.5 * span, 0.5 * span, npt) if npt > 1 else np.array([0.001])
    if shuffle:
        t = rng.permutation(t)
    om = oracle.OracleRR(law)
    om.set_data(t, nsamples=nss, exptimes=0.01 if nss > 1 else 0.0)
    pop = wl.pop
    ldc = np.stack([pop['u1'], pop['u2']], 1) if law == 'quadratic' else rng.uniform(0.4, 0.8, (npv, 2))
    args = [pop['k'], ldc.reshape(npv, 1, 2), pop['t0'], pop['p'], pop['a'], pop['i']]
    f = om.evaluate(args[0][:1, None], args[1][:1], args[2][:1, None], *[x[:1] for x in args[3:]])
    obs = np.atleast_1d(np.squeeze(f)) + rng.normal(0, SIGMA, npt)
    tm = {prec: RoadRunnerModel(law, precision=prec) for prec in ('fp64', 'mixed')}
    for m in tm.values():
        m.set_data(t, nsamples=nss, exptimes=0.01 if nss > 1 else 0.0)
    return om, tm, obs, args


def oracle_lnl(om, obs, args, rows):
    """lnL, and what 1 ppm on every point can move it by."""
    k, ldc, t0, p, a, i = (x[rows] for x in args)
    f = np.atleast_2d(om.evaluate(k[:, None], ldc, t0[:, None], p, a, i)).reshape(len(rows), -1)
    r = (obs[None, :] - f) / SIGMA
    lnl = (-math.log(SIGMA) - 0.5 * math.log(2 * math.pi) - 0.5 * r ** 2).sum(1)
    return lnl, 1e-6 * np.abs(r).sum(1) / SIGMA


# npt: one point, a tile and its neighbours, several splits; nss against the lanes that
# share a point; a long light curve most of whose tiles are outside the window
@pytest.mark.parametrize('npv,npt,nss,law,shuffle,span', [
    (3, 1, 1, 'quadratic', False, 0.4), (2, 255, 3, 'quadratic', False, 0.4), (5, 257, 10, 'power-2', False, 0.4),
    (1, 5000, 5, 'quadratic', False, 0.4), (7, 4097, 20, 'power-2', False, 3.0), (9, 3000, 2, 'quadratic', True, 0.4),
    (1100, 1500, 5, 'quadratic', False, 0.4), (4, 20000, 1, 'quadratic', False, 40.0)])
def test_lnlike_sizes(gpu, oracle, npv, npt, nss, law, shuffle, span):
    om, tm, obs, args = make(oracle, npv, npt, nss, law, npv + npt, shuffle, span)
    rows = np.arange(npv) if npv < 20 else np.array([0, 7, npv - 1])
    ref, ppm = oracle_lnl(om, obs, args, rows)
    for prec in ('fp64', 'mixed'):
        plain = tm[prec].lnlike(*args, obs, SIGMA)
        both, grad = tm[prec].lnlike(*args, obs, SIGMA, grad=True)
        bar = 1e-12 * np.abs(ref) if prec == 'fp64' else ppm
        assert (np.abs(plain[rows] - ref) <= bar).all() and (np.abs(both[rows] - ref) <= bar).all()
        assert np.isfinite(grad).all() and grad.shape == (npv, 7)


def test_lnlike_inputs_in_place(gpu, oracle):
    """Columns of one tensor, plain numbers and host arrays give the same bits."""
    om, tm, obs, args = make(oracle, 40, 2000, 5, 'quadratic', 3)
    k, ldc, t0, p, a, i = args
    ref, gref = tm['fp64'].lnlike(*args, obs, SIGMA, grad=True)
    th = torch.as_tensor(np.stack([k, t0, p, a, i, ldc[:, 0, 0], ldc[:, 0, 1]], 1), device=gpu)
    zero = torch.zeros(40, dtype=torch.float64, device=gpu)
    dev_obs = torch.as_tensor(obs, device=gpu)
    for e, sigma in ((0.0, SIGMA), (zero, torch.full((40,), SIGMA, dtype=torch.float64, device=gpu)),
                     (np.zeros(40), np.array([SIGMA]))):
        lnl, g = tm['fp64'].lnlike(th[:, 0:1], th[:, None, 5:7], th[:, 1], th[:, 2], th[:, 3], th[:, 4], dev_obs, sigma,
                                   e=e, grad=True)
        assert np.array_equal(lnl, ref) and np.array_equal(g, gref)
    # numbers for every parameter but the period
    one = tm['fp64'].lnlike(float(k[0]), ldc[:1], float(t0[0]), np.full(40, p[0]), float(a[0]), float(i[0]), obs, SIGMA)
    assert np.array_equal(one, np.full(40, one[0])) and one[0] == ref[0]
    with pytest.raises(ValueError):
        tm['fp64'].lnlike(th[:3, 0], ldc, t0, p, a, i, obs, SIGMA)
    with pytest.raises(ValueError):
        tm['fp64'].lnlike(np.stack([k, k], 1), ldc, t0, p, a, i, obs, SIGMA)
