"""The window kernel (window_flux.hpp) at the edges of its tiles, chunks and item
arrays, for each model that runs on it, against the FP64 oracle.

Every model is evaluated in FP64 with the oracle's formulas; the kernels differ from
them in the order of a few roundings, so the bar is the suite's FP64 bar, 1e-9
absolute on fluxes of order one; the mixed-precision RoadRunner path has its own bar,
1 ppm.
"""
import numpy as np
import pytest

from pytransit_amd import EclipseModel, OblatePlanetModel, QuadraticModel, RoadRunnerModel, workloads

pytestmark = pytest.mark.gpu

TOL = 1e-9


def layout(name, npt, rng):
    """set_data arguments: times within a transit's reach, so tiles hold points inside
    and outside the window."""
    t = np.linspace(-0.17, 0.21, npt) if npt > 1 else np.array([0.004])
    if name == 'one':
        return dict(time=t, lcids=np.zeros(npt, int), pbids=np.array([0]), nsamples=np.array([5]),
                    exptimes=np.array([0.02]), epids=np.array([0]))
    if name == 'many samples':       # more samples than a chunk's item arrays hold
        return dict(time=t, lcids=np.zeros(npt, int), pbids=np.array([0]), nsamples=np.array([1100]),
                    exptimes=np.array([0.02]), epids=np.array([0]))
    nlc = 4
    lcids = (np.arange(npt) * nlc) // npt
    lcids[:min(npt, nlc)] = np.minimum(lcids[:min(npt, nlc)], nlc - 1)
    ns, ex = np.array([1, 10, 3, 7]), np.array([0.0, 0.02, 0.01, 0.015])
    if name == 'uneven beyond':      # one light curve above the item arrays
        ns = np.array([2, 1, 1030, 4])
    if name == 'shuffled':           # light curves interleaved, times out of order
        order = rng.permutation(npt)
        t, lcids = t[order], lcids[rng.permutation(npt)]
    lcids[:nlc] = np.arange(nlc) if name == 'shuffled' else lcids[:nlc]
    return dict(time=t, lcids=lcids, pbids=np.array([0, 1, 0, 1]), nsamples=ns, exptimes=ex,
                epids=np.array([0, 1, 1, 0]))


CASES = [('one', 1, 3), ('one', 255, 3), ('one', 257, 3), ('one', 1500, 2), ('sorted', 600, 3), ('sorted', 1025, 2),
         ('shuffled', 700, 3), ('many samples', 40, 2), ('uneven beyond', 90, 2),
         ('one', 1027, 1030), ('sorted', 1100, 1030),
         # several sub-tiles a workgroup
         ('one', 9001, 1030), ('sorted', 9001, 1030), ('shuffled', 9001, 1030)]


def population(npv, rng, pb):
    wl = workloads.rr_small(npv=npv, npt=4, seed=int(rng.integers(1000)))
    k = wl.k if pb == 1 else np.concatenate([wl.k, wl.k * 1.03], 1)
    t0 = wl.t0 if pb == 1 else np.concatenate([wl.t0, wl.t0 + 0.01], 1)
    return wl, k, t0


def rows(npv):
    return np.arange(npv) if npv < 20 else np.array([0, 1, npv // 2, npv - 2, npv - 1])


@pytest.mark.parametrize('name,npt,npv', CASES)
def test_mandel_agol(gpu, oracle, name, npt, npv):
    rng = np.random.default_rng(npt + npv)
    d = layout(name, npt, rng)
    pb = int(d['pbids'].max()) + 1
    wl, k, t0 = population(npv, rng, pb)
    k[0], wl.i[0] = 0.5, 0.5 * np.pi       # the special radius ratio, a central transit
    ldc = rng.uniform(0.1, 0.4, (npv, 2 * pb))
    tm = QuadraticModel()
    tm.set_data(**d)
    f = np.atleast_2d(tm.evaluate(k, ldc, t0, wl.p, wl.a, wl.i)).reshape(npv, npt)
    r = rows(npv)
    ref = oracle.quadratic_model(d['time'], k[r], t0[r], wl.p[r], wl.a[r], wl.i[r], wl.e[r], wl.w[r], ldc[r],
                                 d['lcids'], d['pbids'], d['epids'], d['nsamples'], d['exptimes'])
    assert (ref < 1).any()
    assert np.abs(f[r] - ref).max() <= TOL


@pytest.mark.parametrize('name,npt,npv', CASES)
def test_eclipse(gpu, name, npt, npv):
    from oracle import ec_oracle as eo
    rng = np.random.default_rng(npt + 2 * npv)
    d = layout(name, npt, rng)
    d['time'] = d['time'] + 1.01            # around p / 2
    pb = int(d['pbids'].max()) + 1
    wl, k, t0 = population(npv, rng, pb)
    k = k[:, 0].copy()
    k[0] = 0.4
    p = rng.uniform(1.9, 2.1, npv)
    rstar = rng.uniform(0.8, 1.2, npv)
    em = EclipseModel()
    em.set_data(**d)
    f = np.atleast_2d(em.evaluate(k, t0, p, wl.a, wl.i, rstar=rstar)).reshape(npv, npt)
    for j in rows(npv):
        # the model takes passband indices where the kernel takes epoch indices
        ref = eo.eclipse_model(d['time'], k[j:j + 1], t0[j:j + 1], p[j:j + 1], wl.a[j:j + 1], wl.i[j:j + 1],
                               wl.e[j:j + 1], wl.w[j:j + 1], rstar[j], d['pbids'].size, d['lcids'], d['pbids'],
                               d['nsamples'], d['exptimes'])
        assert np.abs(f[j] - ref[0]).max() <= TOL


@pytest.mark.parametrize('name,npt,npv', CASES)
def test_oblate(gpu, oracle, name, npt, npv):
    from oracle import ec_oracle as eo
    nlines = 3 if npt == 9001 else 20
    rng = np.random.default_rng(npt + 3 * npv)
    d = layout(name, npt, rng)
    pb = int(d['pbids'].max()) + 1
    wl, k, t0 = population(npv, rng, pb)
    f, alpha = rng.uniform(0.0, 0.4, npv), rng.uniform(-1.5, 1.5, npv)
    ldc = rng.uniform(0.1, 0.4, (npv, pb, 2))
    m = OblatePlanetModel('quadratic', nlines=nlines)
    m.set_data(**d)
    got = np.atleast_2d(m.evaluate(k, f, alpha, ldc, t0, wl.p, wl.a, wl.i)).reshape(npv, npt)
    ze, zm = oracle.create_z_grid(0.7, 20, 20)
    dk, dg, wt = oracle.weights_3d(256, 0.005, 0.5, ze, 100)
    r = rows(npv)
    ldp, istar = oracle.evaluate_ld('quadratic', oracle.mu_nodes(zm), ldc[r])[:2]
    ref = eo.opmodel(d['time'], k[r], f[r], alpha[r], t0[r], wl.p[r], wl.a[r], wl.i[r], wl.e[r], wl.w[r],
                     d['pbids'].size, pb, 2, nlines, d['lcids'], d['pbids'], d['epids'], d['nsamples'], d['exptimes'],
                     ldp, istar, wt, dk, 0.005, 0.5, dg, ze)
    assert (ref < 1).any()
    assert np.abs(got[r] - ref).max() <= TOL


@pytest.mark.parametrize('precision', ['fp64', 'mixed'])
@pytest.mark.parametrize('name,npt,npv', [c for c in CASES if c[0] not in ('one', 'many samples')])
def test_roadrunner_light_curves(gpu, oracle, name, npt, npv, precision):
    rng = np.random.default_rng(npt + 5 * npv)
    d = layout(name, npt, rng)
    pb = int(d['pbids'].max()) + 1
    wl, k, t0 = population(npv, rng, pb)
    k[0] = (0.3, 0.31)
    if npv > 2:
        wl.a[1] = np.nan                   # an invalid vector, and a passband without a radius
        k[2, 1] = np.nan
    ldc = rng.uniform(0.1, 0.4, (npv, pb, 2))
    om, tm = oracle.OracleRR('quadratic'), RoadRunnerModel('quadratic', precision=precision)
    for m in (om, tm):
        m.set_data(d['time'], d['lcids'], d['pbids'], d['nsamples'], d['exptimes'], d['epids'])
    f = np.atleast_2d(tm.evaluate(k, ldc, t0, wl.p, wl.a, wl.i)).reshape(npv, npt)
    r = rows(npv)
    ref = om.evaluate(np.nan_to_num(k[r], nan=0.1), ldc[r], t0[r], wl.p[r], wl.a[r], wl.i[r], wl.e[r], wl.w[r]).reshape(r.size, npt)
    seen = np.isfinite(k[r]).all(1)        # the reference leaves a NaN radius undefined
    assert np.array_equal(np.isnan(f[r][seen]), np.isnan(ref[seen])) and np.isnan(ref).any() == (npv > 2)
    assert np.nanmin(ref[seen]) < 1
    assert np.nanmax(np.abs(f[r] - ref)[seen]) <= (TOL if precision == 'fp64' else 1e-6)
    if npv > 2:
        assert (f[2][d['pbids'][d['lcids']] == 1] == 1).all()
