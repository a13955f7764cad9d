"""Performance cases: what users of this package compute, through its public models.

A case is a dict of plain values: its ``kind`` (one of ``_KINDS``), the sizes and the
options of the call.  ``prepare`` makes the inputs from a seed and the model that a
user's program keeps (its constructor, ``set_data`` and resident tables), ``run`` is
one evaluation on them, and ``exact`` is the same outputs from plain 64-bit torch
arithmetic, independent of the package's kernels.

The sizes come from the package's workloads (``pytransit_amd/workloads.py``: 64 x
2,000 and 4,096 x 20,000 points for RoadRunner, 1,024 x 512 x 5,000 for transmission
spectroscopy, 2,048 x 10,000 for the gradient, the serving mix) and from its tests,
with ragged sizes between them.
"""
import math

import numpy as np
import torch

BJD = 2459000.0
MIN30 = 30.0 / 1440.0
_LAWS = {'quadratic': 2, 'power-2': 2, 'nonlinear': 4}
_KMIN, _KMAX, _NK, _NG = 0.005, 0.5, 256, 100     # the models' default weight table


def _device():
    return torch.device('cuda', torch.cuda.current_device()) if torch.cuda.is_available() else torch.device('cpu')


# ---------------------------------------------------------------------------- the cases

def listed():
    return [
        # the smallest call: a few walkers on one short light curve (an optimiser's
        # or a small ensemble's step); latency and launches count
        dict(name='population_small', kind='population', law='quadratic', precision='fp64', npv=64, npt=2000,
             nss=1, cadence_s=43.2, pmax=10.0),
        # the package's headline workload: a population over 28 days of 2-min
        # cadence at BJD scale, 30-min exposures supersampled, mixed precision
        dict(name='population_mixed', kind='population', law='power-2', precision='mixed', npv=4096, npt=20000,
             nss=10, cadence_s=120.0, pmax=13.0),
        # the default precision on a ragged size with the four-coefficient law
        dict(name='population_fp64', kind='population', law='nonlinear', precision='fp64', npv=1500, npt=17533,
             nss=5, cadence_s=120.0, pmax=13.0),
        # a joint fit: light curves of several instruments in four passbands with
        # different exposure times and supersampling, eccentric orbits
        dict(name='joint_fit', kind='joint', law='quadratic', precision='fp64', npv=600, npt=9001, nlc=12, npb=4,
             pmax=8.0),
        # a batch of sixteen uneven fit requests through the request server
        dict(name='served_batch', kind='served', precision='mixed', requests=16, npt_max=20000, npv_max=1024,
             npb_max=16),
        # log likelihood of an MCMC ensemble (an LPF's inner loop): no gradient
        dict(name='log_likelihood', kind='likelihood', law='quadratic', precision='fp64', grad=False, npv=250,
             npt=18000, nss=5, span=24.0),
        # log likelihood and its gradient, forward and backward through autograd
        dict(name='gradient', kind='likelihood', law='quadratic', precision='mixed', grad=True, npv=2048, npt=10000,
             nss=5, span=0.7),
        # transmission spectroscopy with tabulated stellar profiles (the largest case)
        dict(name='spectroscopy_mixed', kind='spectroscopy', law='tabulated', precision='mixed', npv=1024, npb=512,
             npt=5000, nss=1),
        # the default precision, a named law, supersampled and ragged
        dict(name='spectroscopy_fp64', kind='spectroscopy', law='quadratic', precision='fp64', npv=100, npb=203,
             npt=1237, nss=3),
        # the Mandel-Agol model of the standard log-posterior functions
        dict(name='mandel_agol', kind='mandel_agol', npv=1000, npt=10007, nss=5, pmax=13.0),
        # secondary eclipses of eccentric planets
        dict(name='eclipse', kind='eclipse', npv=1000, npt=20001, nss=5, pmax=6.0),
        # an oblate planet: 100 scanlines per overlap
        dict(name='oblate', kind='oblate', npv=128, npt=6001, nss=3, nlines=100, pmax=10.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(_KINDS)
    prec = rng.choice(['fp64', 'mixed'])
    if kind == 'population':
        return dict(kind=kind, law=rng.choice(list(_LAWS)), precision=prec, npv=_log_int(rng, 1, 4096),
                    npt=_log_int(rng, 500, 20000), nss=rng.choice([1, 5, 10]), cadence_s=rng.choice([20.0, 43.2, 120.0]),
                    pmax=rng.uniform(5.0, 13.0))
    if kind == 'joint':
        npb = rng.randint(1, 6)
        return dict(kind=kind, law=rng.choice(list(_LAWS)), precision=prec, npv=_log_int(rng, 30, 2000),
                    npt=_log_int(rng, 2000, 20000), nlc=npb * rng.randint(1, 4) + 1, npb=npb, pmax=rng.uniform(4.0, 10.0))
    if kind == 'served':
        return dict(kind=kind, precision=prec, requests=rng.randint(2, 16), npt_max=_log_int(rng, 2000, 20000),
                    npv_max=_log_int(rng, 64, 1024), npb_max=rng.randint(1, 32))
    if kind == 'likelihood':
        return dict(kind=kind, law=rng.choice(['quadratic', 'power-2']), precision=prec, grad=rng.random() < 0.5,
                    npv=_log_int(rng, 16, 2048), npt=_log_int(rng, 500, 20000), nss=rng.choice([1, 5, 10]),
                    span=rng.uniform(0.4, 30.0))
    if kind == 'spectroscopy':
        return dict(kind=kind, law=rng.choice(['tabulated', 'quadratic', 'power-2']), precision=prec,
                    npv=_log_int(rng, 1, 300), npb=_log_int(rng, 8, 512), npt=_log_int(rng, 100, 5000),
                    nss=rng.choice([1, 1, 2, 3, 5]))
    if kind == 'oblate':
        return dict(kind=kind, npv=_log_int(rng, 4, 400), npt=_log_int(rng, 500, 10000), nss=rng.choice([1, 3, 5]),
                    nlines=rng.choice([50, 100, 201]), pmax=rng.uniform(4.0, 12.0))
    return dict(kind=kind, npv=_log_int(rng, 8, 2000), npt=_log_int(rng, 500, 20000), nss=rng.choice([1, 5, 10]),
                pmax=rng.uniform(5.0, 13.0))


_KINDS = ['population', 'joint', 'served', 'likelihood', 'spectroscopy', 'mandel_agol', 'eclipse', 'oblate']


# ------------------------------------------------------------------------------- inputs

def _orbits(rng, npv, pmax, ecc=False):
    """Orbits of a broad population: a from the stellar density, i from the impact parameter."""
    k = rng.uniform(0.05, 0.15, npv)
    p = rng.uniform(1.0, pmax, npv)
    rho = rng.uniform(0.5, 3.0, npv)
    b = rng.uniform(0.0, 0.9, npv)
    t0 = rng.normal(0.0, 0.005, npv)
    a = (6.6743e-11 / (3 * math.pi)) ** (1 / 3) * ((p * 86400.0) ** 2 * 1e3 * rho) ** (1 / 3)
    e = rng.uniform(0.0, 0.3, npv) if ecc else np.zeros(npv)
    w = rng.uniform(0.0, 2 * math.pi, npv) if ecc else np.zeros(npv)
    return dict(k=k, t0=t0, p=p, a=a, i=np.arccos(b / a), e=e, w=w)


def _coefficients(rng, law, npv, npb):
    if law == 'quadratic':
        return np.stack([rng.uniform(0.1, 0.6, (npv, npb)), rng.uniform(0.0, 0.3, (npv, npb))], -1)
    if law == 'power-2':
        return np.stack([rng.uniform(0.3, 0.9, (npv, npb)), rng.uniform(0.3, 1.0, (npv, npb))], -1)
    return np.array([0.56, -0.08, 0.67, -0.33]) + rng.normal(0.0, 0.02, (npv, npb, 4))


def _one_lc(npt):
    return dict(lcids=np.zeros(npt, int), pbids=np.zeros(1, int), epids=np.zeros(1, int))


def _joint_data(rng, case):
    """Contiguous light curves over a month: some long and finely sampled, some short
    with 30-min exposures; the passbands in turn."""
    npt, nlc = case['npt'], case['nlc']
    cuts = np.sort(rng.choice(np.arange(1, npt // 50), nlc - 1, replace=False)) * 50
    size = np.diff(np.concatenate([[0], cuts, [npt]]))
    times, lcids = [], []
    for j, n in enumerate(size):
        start = BJD + rng.uniform(0.0, 30.0)
        times.append(start + np.arange(n) * rng.choice([20.0, 60.0, 120.0]) / 86400.0)
        lcids.append(np.full(n, j))
    nss = rng.choice([1, 5, 10], nlc)
    return dict(times=np.concatenate(times), lcids=np.concatenate(lcids), pbids=np.arange(nlc) % case['npb'],
                epids=np.zeros(nlc, int), nss=nss, exp=np.where(nss > 1, MIN30 * nss / 10.0, 0.0))


def _inputs(case, seed):
    """The call's inputs as numpy arrays, from the seed alone."""
    rng = np.random.default_rng(seed)
    kind = case['kind']
    if kind in ('population', 'mandel_agol', 'eclipse', 'oblate'):
        npv, npt, nss = case['npv'], case['npt'], case['nss']
        s = _orbits(rng, npv, case['pmax'], ecc=kind == 'eclipse')
        s['t0'] = s['t0'] + BJD
        s['times'] = BJD - 0.25 + np.arange(npt) * case.get('cadence_s', 120.0) / 86400.0
        s.update(_one_lc(npt), nss=np.array([nss]), exp=np.array([MIN30 if nss > 1 else 0.0]))
        if kind != 'eclipse':
            s['ldc'] = _coefficients(rng, case.get('law', 'quadratic'), npv, 1)
        if kind == 'eclipse':
            s['rstar'] = rng.uniform(0.7, 1.5, npv)
        if kind == 'oblate':
            s['f'], s['alpha'] = rng.uniform(0.0, 0.2, npv), rng.uniform(0.0, math.pi, npv)
        return s
    if kind == 'joint':
        s = _orbits(rng, case['npv'], case['pmax'], ecc=True)
        s['t0'] = s['t0'] + BJD
        s.update(_joint_data(rng, case), ldc=_coefficients(rng, case['law'], case['npv'], case['npb']))
        return s
    if kind == 'served':
        # the mix of sizes is the case's; the seed gives the parameters
        sizes = np.random.default_rng([case[n] for n in ('requests', 'npt_max', 'npv_max', 'npb_max')])
        datasets = []
        for _ in range(4):
            npt = int(round(math.exp(sizes.uniform(math.log(1000), math.log(case['npt_max'])))))
            npb, nss = int(sizes.integers(1, case['npb_max'] + 1)), int(sizes.choice([1, 5, 10]))
            datasets.append(dict(times=BJD + np.arange(npt) * 120.0 / 86400.0, lcids=(np.arange(npt) * npb) // npt,
                                 pbids=np.arange(npb), epids=np.zeros(npb, int), nss=np.full(npb, nss),
                                 exp=np.full(npb, MIN30 if nss > 1 else 0.0)))
        reqs = []
        for _ in range(case['requests']):
            d = int(sizes.integers(len(datasets)))
            npb = datasets[d]['pbids'].size
            npv = int(round(math.exp(sizes.uniform(math.log(16), math.log(case['npv_max'])))))
            law = str(sizes.choice(list(_LAWS)))
            r = _orbits(rng, npv, 13.0)
            r['k'] = r['k'][:, None] + 0.002 * np.sin(np.arange(npb) / 8.0)[None, :]
            r.update(dataset=d, law=law, t0=BJD + r['t0'], ldc=_coefficients(rng, law, npv, npb))
            reqs.append(r)
        return dict(datasets=datasets, requests=reqs)
    if kind == 'likelihood':
        # an ensemble around one solution and a noisy light curve of it
        npv, npt, nss = case['npv'], case['npt'], case['nss']
        tr = _orbits(rng, 1, 6.0)
        tr.update(t0=np.array([BJD]), ldc=_coefficients(rng, case['law'], 1, 1),
                  times=BJD - 0.35 + np.arange(npt) * (case['span'] / npt))
        tr.update(_one_lc(npt), nss=np.array([nss]), exp=np.array([0.01 if nss > 1 else 0.0]))
        s = dict(tr)
        for name, sig in (('k', 2e-3), ('t0', 1e-3), ('p', 1e-4), ('a', 0.05), ('i', 2e-3)):
            s[name] = tr[name] + rng.normal(0.0, sig, npv)
        s['i'] = np.minimum(s['i'], 0.5 * math.pi)
        s['e'], s['w'] = np.zeros(npv), np.zeros(npv)
        s['ldc'] = tr['ldc'] + rng.normal(0.0, 0.02, (npv, 1, 2))
        s['sigma'] = 300e-6
        flux = _rr_flux(_on(tr, torch.device('cpu')), case['law'])[0].numpy()
        s['obs'] = flux + rng.normal(0.0, s['sigma'], npt)
        return s
    # spectroscopy: radius ratios and limb darkening varying smoothly with wavelength
    npv, npb, npt, nss = (case[n] for n in ('npv', 'npb', 'npt', 'nss'))
    s = _orbits(rng, npv, 10.0)
    x = np.arange(npb) * (512.0 / npb)
    s['k'] = rng.uniform(0.08, 0.12, npv)[:, None] + 0.002 * np.sin(x / 40.0)[None, :]
    s['times'] = np.linspace(-0.2, 0.2, npt)
    s.update(_one_lc(npt), nss=np.array([nss]), exp=np.array([120.0 / 86400.0 if nss > 1 else 0.0]))
    if case['law'] == 'power-2':
        s['ldc'] = _coefficients(rng, 'power-2', npv, npb)
    else:
        s['ldc'] = np.stack([0.55 - 0.25 * x / 511.0 + rng.normal(0.0, 0.01, (npv, npb)),
                             0.25 - 0.10 * x / 511.0 + rng.normal(0.0, 0.01, (npv, npb))], -1)
    return s


def _on(s, dev):
    return {n: torch.as_tensor(v, device=dev) if isinstance(v, np.ndarray) else v for n, v in s.items()}


def _table_profiles(s, mu):
    """Tabulated profiles [npv, npb, nmu] and their disk integrals from quadratic coefficients."""
    x = 1.0 - mu
    u1, u2 = s['ldc'][..., 0:1], s['ldc'][..., 1:2]
    return 1.0 - u1 * x - u2 * x ** 2, math.pi / 6 * (6.0 - 2.0 * u1[..., 0] - u2[..., 0])


def prepare(case, seed):
    from pytransit_amd import (EclipseModel, OblatePlanetModel, QuadraticModel, RoadRunnerModel, TabulatedLDModel,
                               TSModel)
    from pytransit_amd.lpf import RoadRunnerLPFModel
    from pytransit_amd.serving import Dataset, RRServer

    kind = case['kind']
    raw = _inputs(case, seed)
    if kind == 'served':
        server = RRServer(hbm_budget=4 << 30, precision=case['precision'], staging_bytes=16 << 20)
        dsets = [Dataset(d['times'], d['lcids'], d['pbids'], d['nss'], d['exp'], d['epids']) for d in raw['datasets']]
        reqs = [((dsets[r['dataset']], r['k'], r['ldc'], r['t0'], r['p'], r['a'], r['i']), r['law'])
                for r in raw['requests']]
        return dict(kind=kind, server=server, requests=reqs, last=[])
    s = _on({n: v for n, v in raw.items() if n not in ('times', 'lcids', 'pbids', 'epids', 'nss', 'exp')}, _device())
    data = (raw['times'], raw['lcids'], raw['pbids'], raw['nss'], raw['exp'], raw['epids'])
    k, t0 = s['k'], s['t0']
    orbit = (s['p'], s['a'], s['i'], s['e'], s['w'])
    if kind in ('population', 'joint'):
        model = RoadRunnerModel(case['law'], precision=case['precision'])
        args = (k[:, None], s['ldc'], t0[:, None]) + orbit
    elif kind == 'likelihood' and case['grad']:
        model = RoadRunnerModel(case['law'], precision=case['precision'])
        theta = torch.cat([torch.stack([k, t0, s['p'], s['a'], s['i']], 1), s['ldc'][:, 0]], 1).requires_grad_()
        args = (theta, model, s['obs'], s['sigma'])
    elif kind == 'likelihood' and case['law'] == 'quadratic':
        model = RoadRunnerLPFModel(precision=case['precision'])
        args = (k, s['ldc'][:, 0].contiguous(), t0) + orbit[:3] + (s['obs'], s['sigma'])
    elif kind == 'likelihood':
        model = RoadRunnerModel(case['law'], precision=case['precision'])
        args = (k, s['ldc'], t0) + orbit[:3] + (s['obs'], s['sigma'])
    elif kind == 'spectroscopy':
        if case['law'] == 'tabulated':
            mu = torch.as_tensor(_z_grid(64, 64)[1], device=_device())
            model = TSModel(TabulatedLDModel(*_table_profiles(s, mu)), nzin=64, nzlimb=64, precision=case['precision'])
            args = (k, None, t0) + orbit
        else:
            model = TSModel(case['law'], precision=case['precision'])
            args = (k, s['ldc'], t0) + orbit
    elif kind == 'mandel_agol':
        model = QuadraticModel()
        args = (k, s['ldc'][:, 0].contiguous(), t0) + orbit
    elif kind == 'eclipse':
        model = EclipseModel()
        args = (k, t0) + orbit + (s['rstar'],)
    else:
        model = OblatePlanetModel('quadratic', nlines=case['nlines'])
        args = (k[:, None], s['f'], s['alpha'], s['ldc'], t0[:, None]) + orbit
    model.set_data(*data)
    if hasattr(model, 'weights'):
        model.weights      # the weight table, built once per model and device
    return dict(kind=kind, model=model, args=args, grad=case.get('grad', False))


def run(state):
    kind = state['kind']
    if kind == 'served':
        for r in state['last']:
            r.release()
        server = state['server']
        state['last'] = [server.submit(*args, ld=law) for args, law in state['requests']]
        server.run()
        server.completed.clear()
        return [r.result(copy=False) for r in state['last']]
    model, args = state['model'], state['args']
    if kind == 'likelihood':
        if state['grad']:
            from pytransit_amd.autograd import rr_lnlike
            lnl = rr_lnlike(*args)
            grad, = torch.autograd.grad(lnl.sum(), args[0])
            return lnl.detach(), grad
        if hasattr(model, 'lnlikelihood'):
            return model.lnlikelihood(*args, copy=False)
        return model.lnlike(*args, copy=False)
    return model.evaluate(*args, copy=False)


# --------------------------------------------------------------------------------- work

def _duty(pmax):
    """Mean share of the time in transit of _orbits' draws."""
    p = np.linspace(1.0, pmax, 64)
    a = 4.2083 * p ** (2 / 3) * 1.75 ** (1 / 3)
    return float(np.mean(np.sqrt(1.1 ** 2 - 0.27) / (math.pi * a)))


def work(case):
    kind = case['kind']
    if kind == 'served':
        # sixteen or fewer requests of log-uniform sizes
        mean = lambda lo, hi: (hi - lo) / math.log(hi / lo)   # noqa: E731
        pts = case['requests'] * mean(1000, case['npt_max'] + 1) * mean(16, case['npv_max'] + 1)
        return dict(bytes=pts * (4 if case['precision'] == 'mixed' else 8), flops=pts * _duty(13.0) * 5 * 60)
    npv, npt, nss = case['npv'], case['npt'], case.get('nss', 5)
    real = 4 if case.get('precision') == 'mixed' else 8
    pts = npv * npt
    if kind == 'spectroscopy':
        npb = case['npb']
        ngz = _NG * (128 if case['law'] == 'tabulated' else 40)
        read = npv * npb * (8 * 129 if case['law'] == 'tabulated' else 24) + 8 * npt
        return dict(bytes=pts * npb * real + read, flops=0.4 * pts * (60 + 6 * npb) * nss + 2 * npv * npb * ngz)
    if kind == 'likelihood':
        duty = min(0.5, 0.15 / case['span'] + _duty(6.0))
        return dict(bytes=16 * npt + npv * 8 * (15 if case['grad'] else 8),
                    flops=npv * duty * npt * nss * (200 if case['grad'] else 60))
    per_sample = {'mandel_agol': 250, 'oblate': 60 + 2 * case.get('nlines', 0)}.get(kind, 60)
    return dict(bytes=pts * real + 8 * npt + npv * 80, flops=pts * _duty(case['pmax']) * nss * per_sample)


# -------------------------------------------------- the same in plain 64-bit arithmetic

def _z_grid(nin, nlimb, zcut=0.7):
    """Annulus edges, uniform in z to zcut and in mu from there to the limb, and the mu nodes."""
    n = nin + nlimb
    ze, zm = np.zeros(n), np.zeros(n)
    ze[:nin - 1] = np.arange(1, nin) * (zcut / nin)
    ze[n - 1 - np.arange(nlimb + 1)] = np.sqrt(1.0 - (np.arange(nlimb + 1) * (math.sqrt(1.0 - zcut ** 2) / nlimb)) ** 2)
    zm[1:] = 0.5 * (ze[:-1] + ze[1:])
    return ze, np.sqrt(1.0 - zm ** 2)


def _weights(k, ze):
    """Shares of each annulus in the planet's disk, [len(k), ng, nz], on the grid of grazing parameters."""
    g = torch.as_tensor(np.linspace(0.0, 1.0 - 1e-7, _NG), device=k.device)
    r, k = ze[None, None, :], k[:, None, None]
    b = (g[None, :, None] * (1.0 + k)).expand(-1, -1, ze.numel())
    none, whole, ring = r < b - k, r >= b + k, b - k <= -r
    lens = ~(none | whole | ring)
    bs = torch.where(lens, b, 1.0)
    area = (k * k * torch.acos(torch.where(lens, (b * b + k * k - r * r) / (2 * bs * k), 0.0)) +
            r * r * torch.acos(torch.where(lens, (b * b + r * r - k * k) / (2 * bs * r), 0.0)) -
            0.5 * torch.sqrt(torch.where(lens, (-b + k + r) * (b + k - r) * (b - k + r) * (b + k + r), 0.0)))
    area = torch.where(none, 0.0, torch.where(whole, math.pi * k * k, torch.where(ring, math.pi * r * r, area)))
    wt = torch.diff(area, dim=-1, prepend=torch.zeros_like(area[..., :1]))
    return wt / wt.sum(-1, keepdim=True)


def _law(law, mu, c):
    """Intensity at mu for coefficients c[..., nldc]."""
    c = [c[..., j:j + 1] for j in range(c.shape[-1])]
    if law == 'quadratic':
        return 1.0 - c[0] * (1.0 - mu) - c[1] * (1.0 - mu) ** 2
    if law == 'power-2':
        return 1.0 - c[0] * (1.0 - mu ** c[1])
    return (1.0 - c[0] * (1.0 - mu ** 0.5) - c[1] * (1.0 - mu) - c[2] * (1.0 - mu ** 1.5) - c[3] * (1.0 - mu ** 2))


def _disk_integral(law, c):
    if law == 'quadratic':
        return math.pi / 6 * (6.0 - 2.0 * c[..., 0] - c[..., 1])
    if law == 'power-2':
        return 2 * math.pi * (-c[..., 0] * c[..., 1] + c[..., 1] + 2.0) / (2.0 * c[..., 1] + 4.0)
    mu = torch.as_tensor(np.linspace(1.0, 0.0, 200), device=c.device)
    z = torch.sqrt(1.0 - mu * mu)
    return 2 * math.pi * torch.trapezoid(z * _law(law, mu, c), z, dim=-1)


def _conjunction(e, w, at):
    """Mean anomaly at true anomaly at - w."""
    ea = torch.atan2(torch.sqrt(1.0 - e * e) * torch.sin(at - w), e + torch.cos(at - w))
    return ea - e * torch.sin(ea)


def _taylor(s, shift=None):
    """Coefficients [npv, 5] of x and y in powers of the time from mid-transit (or `shift`
    later): central differences over seven Kepler positions 0.02 d apart."""
    p, a, i, e, w = (s[n][:, None] for n in ('p', 'a', 'i', 'e', 'w'))
    h = 0.02
    t = torch.arange(-3, 4, device=p.device, dtype=torch.float64)[None, :] * h
    t = t if shift is None else t + shift[:, None]
    m = torch.remainder(2 * math.pi * t / p + _conjunction(e, w, 0.5 * math.pi), 2 * math.pi)
    ea = m.detach()
    for _ in range(60):
        ea = ea - (ea - e.detach() * torch.sin(ea) - m.detach()) / (1.0 - e.detach() * torch.cos(ea))
    ea = ea - (ea - e * torch.sin(ea) - m) / (1.0 - e * torch.cos(ea))   # carries the derivatives
    f = torch.atan2(torch.sqrt(1.0 - e * e) * torch.sin(ea), torch.cos(ea) - e)
    r = a * (1.0 - e * e) / (1.0 + e * torch.cos(f))
    out = []
    for j, q in enumerate((-r * torch.cos(w + f), -r * torch.sin(w + f) * torch.cos(i))):
        q0, q1, q2, q3, q4, q5, q6 = q.unbind(1)
        v = ((q6 - q0) + 9 * (q1 - q5) + 45 * (q4 - q2)) / 60 / h
        acc = ((q0 + q6) / 90 - 0.15 * (q1 + q5) + 1.5 * (q2 + q4) - 49 / 18 * q3) / h ** 2
        jerk = ((q0 - q6) / 8 + (q5 - q1) + 13 / 8 * (q2 - q4)) / h ** 3
        snap = (-(q0 + q6) / 6 + 2 * (q1 + q5) - 6.5 * (q2 + q4) + 28 / 3 * q3) / h ** 4
        out.append(torch.stack([torch.zeros_like(q3) if j == 0 else q3, v, acc / 2, jerk / 6, snap / 24], 1))
    return out


def _poly(c, t):
    return (((c[..., 4] * t + c[..., 3]) * t + c[..., 2]) * t + c[..., 1]) * t + c[..., 0]


def _contacts(k, c):
    """First and fourth contact about the series' origin, by bisection."""
    found = []
    v = c[0][:, 1].abs()
    for side in (-1.0, 1.0):
        lo, hi = torch.zeros_like(v), side * 2.0 / v
        for _ in range(48):
            mid = 0.5 * (lo + hi)
            out = torch.hypot(_poly(c[0], mid), _poly(c[1], mid)) > 1.0 + k
            lo, hi = torch.where(out, lo, mid), torch.where(out, mid, hi)
        found.append(0.5 * (lo + hi))
    return found


def _lens(k, z):
    """Area of a disk of radius k < 1 on the unit disk at separation z, and half the angle it
    is seen over from its own centre (kappa_0)."""
    part = (z > 1.0 - k) & (z < 1.0 + k)
    zz = torch.where(part, z, 1.0)
    prod = (1.0 + k + zz) * (k - (1.0 - zz)) * (k + (1.0 - zz)) * (1.0 + zz - k)
    kite = torch.sqrt(torch.where(part, prod, 1.0))
    k0 = torch.atan2(kite, (k - 1.0) * (k + 1.0) + zz * zz)
    k1 = torch.atan2(kite, (1.0 - k) * (1.0 + k) + zz * zz)
    full = z <= 1.0 - k
    area = torch.where(part, k1 + k * k * k0 - 0.5 * kite, torch.where(full, math.pi * k * k, 0.0))
    return area, torch.where(part, k0, math.pi * full.to(z.dtype))


def _means(s, law, nz=(20, 20)):
    """Mean limb darkening under the planet [npv, npb, ng] from the table in k, and I*."""
    dev = s['ldc'].device
    ze, mu = (torch.as_tensor(x, device=dev) for x in _z_grid(*nz))
    ks = torch.as_tensor(np.linspace(_KMIN, _KMAX, _NK), device=dev)
    k0 = s['k'][:, 0] if s['k'].dim() == 2 else s['k']
    dk = (_KMAX - _KMIN) / _NK
    ik = torch.clamp(torch.floor((k0.detach() - _KMIN) / dk), max=_NK - 2)
    ak = ((k0 - _KMIN - ik * dk) / dk)[:, None, None]
    rows, back = torch.unique(ik.long(), return_inverse=True)
    w0, w1 = _weights(ks[rows], ze)[back], _weights(ks[rows + 1], ze)[back]
    ldp = _law(law, mu, s['ldc'])
    wt = (1.0 - ak) * w0 + ak * w1
    return torch.matmul(ldp, wt.transpose(1, 2).contiguous()), _disk_integral(law, s['ldc'])


def _interpolate(ldm, row, z, k):
    """Rows `row` of ldm[rows, ng] at the grazing parameter z / (1 + k)."""
    dg = (1.0 - 1e-7) / (_NG - 1)
    g = z / (1.0 + k)
    j = torch.clamp(torch.floor(g.detach() / dg), 0, _NG - 2)
    al = (g - j * dg) / dg
    at = (row * _NG)[:, None] + j.long() if row.dim() < g.dim() else row * _NG + j.long()
    flat = ldm.reshape(-1)
    return torch.where(g <= 1.0, (1.0 - al) * flat[at] + al * flat[at + 1], 0.0)


def _in_window(s, lo, hi, te, margin, rows):
    """(ipv, it, time from mid-transit) of the points in the window, for the rows of a chunk."""
    lc = s['lcids']
    p = s['p'][rows][:, None]
    tz = te[rows][:, None]
    epoch = torch.floor((s['times'][None, :] - tz + 0.5 * p) / p).detach()
    tc = s['times'][None, :] - (tz + epoch * p)
    m = (margin + s['exp'])[lc][None, :]
    ipv, it = torch.nonzero((lo[rows][:, None] - m <= tc) & (tc <= hi[rows][:, None] + m), as_tuple=True)
    return ipv, it, tc[ipv, it]


def _by_sampling(s, ipv, it):
    """Groups of in-window points with one nsamples: (selection, sample times from mid-exposure)."""
    ns = s['nss'][s['lcids'][it]]
    for n in torch.unique(ns).tolist():
        sel = torch.nonzero(ns == n)[:, 0]
        off = (torch.arange(n, device=it.device, dtype=torch.float64) + 0.5) / n - 0.5
        yield sel, s['exp'][s['lcids'][it[sel]]][:, None] * off[None, :]


def _chunks(npv, npt, most=1 << 23):
    step = max(1, most // max(1, npt))
    return [slice(j, min(npv, j + step)) for j in range(0, npv, step)]


def _rr_flux(s, law):
    """The RoadRunner flux [npv, npt]."""
    npv, npt, npb = s['p'].numel(), s['times'].numel(), s['ldc'].shape[1]
    c = _taylor(s)
    k = s['k'] if s['k'].dim() == 2 else s['k'][:, None]
    lo, hi = _contacts(k[:, 0], c)
    ldm, ist = _means(s, law)
    out = torch.ones((npv, npt), dtype=torch.float64, device=s['p'].device)
    for rows in _chunks(npv, npt):
        ipv, it, tc = _in_window(s, lo, hi, s['t0'], 0.003, rows)
        ipv = ipv + rows.start
        for sel, off in _by_sampling(s, ipv, it):
            q, t = ipv[sel], tc[sel][:, None] + off
            pb = s['pbids'][s['lcids'][it[sel]]]
            kq = k[q, pb if k.shape[1] > 1 else 0][:, None]
            z = torch.hypot(_poly(c[0][q][:, None], t), _poly(c[1][q][:, None], t))
            depth = _interpolate(ldm, q * npb + pb, z, kq) * _lens(kq, z)[0]
            out[q, it[sel]] = (1.0 - depth / ist[q, pb][:, None]).mean(1)
    return out


def _exact_likelihood(s, law, grad):
    npv, npt = s['p'].numel(), s['times'].numel()
    lnl, grads = [], []
    for rows in _chunks(npv, npt, 1 << 21):
        r = {n: s[n] for n in ('times', 'lcids', 'pbids', 'epids', 'nss', 'exp')}
        th = torch.cat([torch.stack([s[n][rows] for n in ('k', 't0', 'p', 'a', 'i')], 1), s['ldc'][rows, 0]], 1)
        th.requires_grad_(grad)
        r.update(zip(('k', 't0', 'p', 'a', 'i'), th.unbind(1)), ldc=th[:, None, 5:7], e=s['e'][rows], w=s['w'][rows])
        c = _taylor(r)
        lo, hi = (x.detach() for x in _contacts(r['k'].detach(), [x.detach() for x in c]))
        ldm, ist = _means(r, law)
        q, it, tc = _in_window(r, lo, hi, r['t0'], 0.003, slice(0, th.shape[0]))
        (sel, off), = _by_sampling(r, q, it)
        t = tc[sel][:, None] + off
        kq = r['k'][q][:, None]
        z = torch.sqrt(_poly(c[0][q][:, None], t) ** 2 + _poly(c[1][q][:, None], t) ** 2)
        m = 1.0 - (_interpolate(ldm, q, z, kq) * _lens(kq, z)[0]).mean(1) / ist[q, 0]
        o = s['obs']
        inside = torch.zeros(th.shape[0], dtype=torch.float64, device=th.device).index_add(0, q, (o[it] - m) ** 2)
        away = torch.ones((th.shape[0], npt), dtype=torch.float64, device=th.device)
        away[q, it] = 0.0
        chi = inside + (away * ((o - 1.0) ** 2)[None, :]).sum(1)
        l = -npt * (math.log(s['sigma']) + 0.5 * math.log(2 * math.pi)) - 0.5 * chi / s['sigma'] ** 2
        lnl.append(l.detach())
        if grad:
            grads.append(torch.autograd.grad(l.sum(), th)[0])
    return (torch.cat(lnl), torch.cat(grads)) if grad else torch.cat(lnl)


def _exact_spectroscopy(s, case):
    table = case['law'] == 'tabulated'
    dev = s['p'].device
    ze, mu = (torch.as_tensor(x, device=dev) for x in _z_grid(*((64, 64) if table else (20, 20))))
    km, kmax = s['k'].mean(1), s['k'].max(1).values
    c = _taylor(s)
    lo, hi = _contacts(km, c)
    npv, npb, npt = case['npv'], case['npb'], case['npt']
    out = torch.ones((npv, npb, npt), dtype=torch.float64, device=dev)
    for rows in _chunks(npv, 1, 64):
        wt = _weights(km[rows], ze)
        sub = dict(ldc=s['ldc'][rows])
        ldp, ist = _table_profiles(sub, mu) if table else (_law(case['law'], mu, sub['ldc']),
                                                           _disk_integral(case['law'], sub['ldc']))
        ldm = torch.matmul(ldp, wt.transpose(1, 2).contiguous())     # [rows, npb, ng]
        pts = _in_window(s, lo, hi, s['t0'], 0.0015, rows)
        for j in range(ldm.shape[0]):
            q = rows.start + j
            mine = pts[0] == j
            it, tc = pts[1][mine], pts[2][mine]
            if it.numel() == 0:
                continue
            (sel, off), = _by_sampling(s, pts[0][mine], it)
            t = tc[sel][:, None] + off
            z = torch.hypot(_poly(c[0][q], t), _poly(c[1][q], t))
            area, kap = _lens(km[q], z)
            kq = s['k'][q][:, None, None]
            area = torch.where(z <= 1.0 - kmax[q], area * (kq / km[q]) ** 2, area + (kq - km[q]) * 2.0 * km[q] * kap)
            row = torch.arange(npb, device=dev)[:, None, None]
            ip = _interpolate(ldm[j], row, z[None], km[q])
            out[q][:, it[sel]] = 1.0 - (ip * area).mean(2) / ist[j][:, None]
    return out


def _ell_k(k):
    """K(k) by the polynomial approximation of Abramowitz & Stegun 17.3.34, as the model has it."""
    m = 1.0 - k * k
    a = 1.38629436112 + m * (0.09666344259 + m * (0.03590092383 + m * (0.03742563713 + m * 0.01451196212)))
    b = 0.5 + m * (0.12498593597 + m * (0.06880248576 + m * (0.03328355346 + m * 0.00441787012)))
    return a - b * torch.log(m)


def _ell_e(k):
    """E(k), Abramowitz & Stegun 17.3.36."""
    m = 1.0 - k * k
    a = 1.0 + m * (0.44325141463 + m * (0.06260601220 + m * (0.04757383546 + m * 0.01736506451)))
    b = m * (0.24998368310 + m * (0.09200180037 + m * (0.04069697526 + m * 0.00526449639)))
    return a - b * torch.log(m)


def _ell_pi(n, k):
    """Complete elliptic integral of the third kind (Bulirsch 1965)."""
    kc = torch.sqrt(1.0 - k * k)
    e, p = kc, torch.sqrt(n + 1.0)
    m0, c, d = torch.ones_like(kc), torch.ones_like(kc), 1.0 / p
    done = torch.zeros_like(kc)
    open_ = torch.ones_like(kc, dtype=torch.bool)
    for _ in range(24):
        f, c = c, d / p + c
        g = e / p
        d = 2.0 * (f * g + d)
        p = g + p
        g, m0 = m0, kc + m0
        ready = open_ & ~((1.0 - kc / g).abs() > 1e-8)
        done = torch.where(ready, 0.5 * math.pi * (c * m0 + d) / (m0 * (m0 + p)), done)
        open_ = open_ & ~ready
        kc = 2.0 * torch.sqrt(e)
        e = kc * m0
    return done


def _mandel_agol(z, k, u1, u2):
    """Flux of Mandel & Agol (2002) for 0 < k < 0.5 and z < 1 + k."""
    pi = math.pi
    z = torch.where((z - k).abs() < 1e-6, z + 1e-6, z)
    x1, x2, x3 = (k - z) ** 2, (k + z) ** 2, k * k - z * z
    full = z < 1.0 - k
    edge = (z - k).abs() < 1e-4 * (z + k)
    k1 = torch.acos(((1.0 - k * k + z * z) / (2.0 * z)).clamp(-1.0, 1.0))
    k0 = torch.acos(((k * k + z * z - 1.0) / (2.0 * k * z)).clamp(-1.0, 1.0))
    lune = 0.5 * torch.sqrt((4.0 * z * z - (1.0 + z * z - k * k) ** 2).clamp(min=0.0))
    le = torch.where(z <= 1.0 - k, k * k, (k * k * k0 + k1 - lune) / pi)
    qf = torch.sqrt(torch.where(full, (x2 - x1) / (1.0 - x1), 0.5))
    ldf = 2 / (9 * pi) / torch.sqrt(1.0 - x1) * (
        (1.0 - 5.0 * z * z + k * k + x3 * x3) * _ell_k(qf) + (1.0 - x1) * (z * z + 7.0 * k * k - 4.0) * _ell_e(qf) -
        3.0 * x3 / x1 * _ell_pi(x2 / x1 - 1.0, qf)) + 2 / 3 * (z < k).to(z.dtype)
    touch = 2 / (3 * pi) * torch.acos(1.0 - 2.0 * k) - 4 / (9 * pi) * torch.sqrt(k * (1.0 - k)) * (3.0 + 2.0 * k - 8.0 * k * k)
    ldf = torch.where((k + z - 1.0).abs() < 1e-4, touch, ldf)
    qp = torch.sqrt(torch.where(full, 0.25, (1.0 - x1) / (4.0 * z * k)))
    ldp = 1 / (9 * pi) / torch.sqrt(k * z) * (
        ((1.0 - x2) * (2.0 * x2 + x1 - 3.0) - 3.0 * x3 * (x2 - 2.0)) * _ell_k(qp) +
        4.0 * k * z * (z * z + 7.0 * k * k - 4.0) * _ell_e(qp) - 3.0 * x3 / x1 * _ell_pi(1.0 / x1 - 1.0, qp))
    lde = 1 / 3 + 2 / (9 * pi) * (4.0 * (2.0 * k * k - 1.0) * _ell_e(2.0 * k) + (1.0 - 4.0 * k * k) * _ell_k(2.0 * k))
    ld = torch.where(edge, lde, torch.where(full, ldf, ldp))
    etf = k * k / 2 * (k * k + 2.0 * z * z)
    etp = 1 / (2 * pi) * (k1 + k * k * (k * k + 2.0 * z * z) * k0 -
                          (1.0 + 5.0 * k * k + z * z) / 4 * torch.sqrt(((1.0 - x1) * (x2 - 1.0)).clamp(min=0.0)))
    ed = torch.where(full | edge, etf, etp)
    return 1.0 - ((1.0 - u1 - 2.0 * u2) * le + (u1 + 2.0 * u2) * ld + u2 * ed) / (1.0 - u1 / 3 - u2 / 6)


def _ellipse_area(cx, cy, z, k, f, alpha, ny):
    """Area of the rotated ellipse of semi-axes k and k (1 - f) about (cx, cy) on the unit disk,
    summed over ny rows; 1-d inputs."""
    j = torch.arange(1, ny + 1, device=z.device, dtype=torch.float64)
    y = (j * (2.0 / (ny + 1)) - 1.0)[None, :]
    k, f, ca, sa = k[:, None], f[:, None], torch.cos(alpha)[:, None], torch.sin(alpha)[:, None]
    b = 1.0 - f
    d = b * b * ca * ca + sa * sa - y * y * (ca * ca + sa * sa) ** 2
    row = d >= 0
    d = torch.sqrt(torch.where(row, d, 0.0)) / b
    u, v = ca * sa * y * (1.0 / (b * b) - 1.0), (sa / b) ** 2 + ca * ca
    left, right = k * (u - d) / v, k * (u + d) / v
    h2 = 1.0 - (k * y + cy[:, None]) ** 2
    half = torch.sqrt(h2.clamp(min=0.0))
    a1, a2 = -half - cx[:, None], half - cx[:, None]
    west, east = cx[:, None] < -k, cx[:, None] > k
    mid = torch.minimum(a2, right) - torch.maximum(a1, left)
    wst = (right - torch.maximum(a1, left)).clamp(min=0.0)
    est = (torch.minimum(a2, right) - left).clamp(min=0.0)
    part = torch.where(west, wst, torch.where(east, est, mid))
    part = torch.where(row & (h2 >= 0.0), part, 0.0)
    return part.sum(1) * (k[:, 0] * (2.0 / (ny + 1)))


def _exact_single(s, case):
    """The Mandel-Agol, eclipse and oblate models on one light curve: [npv, npt]."""
    kind, npv, npt = case['kind'], case['npv'], case['npt']
    te, shift = s['t0'], None
    if kind == 'eclipse':
        e, w = s['e'], s['w']
        ph = (_conjunction(e, w, 1.5 * math.pi) - _conjunction(e, w, 0.5 * math.pi)) * s['p'] / (2 * math.pi)
        shift = torch.where(ph > 0.0, ph, s['p'] + ph)
        om = s['a'] * (1.0 - e * e)
        path = (om / (1.0 + e * torch.sin(w)) + om / (1.0 - e * torch.sin(w))) * torch.sin(s['i'])
        te = te + (shift + path * s['rstar'] * 6.957e8 / 299792458.0 / 86400.0)
    c = _taylor(s, shift)
    lo, hi = _contacts(s['k'], c)
    base = math.pi * s['k'] ** 2 if kind == 'eclipse' else torch.ones_like(s['k'])
    out = base[:, None].repeat(1, npt)
    margin = {'mandel_agol': 0.025 - float(s['exp'][0]), 'eclipse': 0.003, 'oblate': 0.0015}[kind]
    if kind == 'oblate':
        ldm, ist = _means(s, 'quadratic')
    for rows in _chunks(npv, npt):
        q, it, tc = _in_window(s, lo, hi, te, margin, rows)
        q = q + rows.start
        for sel, off in _by_sampling(s, q, it):
            j, t = q[sel], tc[sel][:, None] + off
            k = s['k'][j][:, None]
            x, y = _poly(c[0][j][:, None], t), _poly(c[1][j][:, None], t)
            z = torch.hypot(x, y)
            if kind == 'mandel_agol':
                u1, u2 = (s['ldc'][j, 0, m][:, None] for m in (0, 1))
                on = z <= 1.0 + k
                f = torch.where(on, _mandel_agol(torch.where(on, z, 0.5 + 0.0 * z), k, u1, u2), 1.0)
            elif kind == 'eclipse':
                f = math.pi * k * k - _lens(k, z)[0]
            else:
                kk, fl = k.expand_as(z).reshape(-1), s['f'][j][:, None].expand_as(z).reshape(-1)
                al, zz = s['alpha'][j][:, None].expand_as(z).reshape(-1), z.reshape(-1)
                area = torch.where(zz <= 1.0 - kk, math.pi * kk * kk * (1.0 - fl), 0.0)
                cut = torch.nonzero((zz > 1.0 - kk) & (zz < 1.0 + kk))[:, 0]
                for part in torch.split(cut, 1 << 17):
                    area[part] = _ellipse_area(x.reshape(-1)[part], y.reshape(-1)[part], zz[part], kk[part], fl[part],
                                               al[part], case['nlines'])
                f = 1.0 - _interpolate(ldm, j, z, k) * area.reshape(z.shape) / ist[j]
            out[j, it[sel]] = f.mean(1)
    return out


def exact(case, seed):
    raw = _inputs(case, seed)
    kind, dev = case['kind'], _device()
    if kind == 'served':
        return [_rr_flux(_on({**raw['datasets'][r['dataset']], **r}, dev), r['law']) for r in raw['requests']]
    s = _on(raw, dev)
    if kind in ('population', 'joint'):
        return _rr_flux(s, case['law'])
    if kind == 'likelihood':
        return _exact_likelihood(s, case['law'], case['grad'])
    if kind == 'spectroscopy':
        return _exact_spectroscopy(s, case)
    return _exact_single(s, case)
