"""The launches chosen by the density of the times against those without it: the same bits.
Sizes on both sides of each rule: one and four times a lane, one and several sub-tiles a
workgroup, fewer and more than four tiles of a vector."""
import numpy as np
import pytest

from pytransit_amd import EclipseModel, OblatePlanetModel, QuadraticModel, RoadRunnerModel

pytestmark = pytest.mark.gpu


def orbits(npv):
    rng = np.random.default_rng(npv)
    a = rng.uniform(5, 15, npv)
    return (rng.uniform(1, 10, npv), a, np.arccos(rng.uniform(0, 0.9, npv) / a), rng.uniform(0.03, 0.15, npv),
            rng.normal(0, 0.01, npv), np.tile([0.3, 0.2], (npv, 1)), np.zeros(npv))


def both(m, args):
    with_bits = np.array(m.evaluate(*args, copy=True))
    data, = m._dev_data.values()
    assert data['sorted'] >> 8
    data['sorted'] &= 0xff
    return with_bits, np.array(m.evaluate(*args, copy=True))


# times in a tenth of a day / samples: P and sub-tiles a workgroup differ with and without the bits
@pytest.mark.parametrize('npv,npt,span', [(700, 3073, 3.0), (700, 3073, 0.3), (350, 20011, 2.0), (40, 3000, 0.3)])
@pytest.mark.parametrize('ns', [1, 5, 20, (2, 30)])
@pytest.mark.parametrize('kind', ['ma', 'ec', 'op'])
def test_window_models(gpu, npv, npt, span, ns, kind):
    p, a, inc, k, t0, ldc, z = orbits(npv)
    t = np.linspace(-span / 3, span, npt)
    ids = np.repeat([0, 1], [npt // 3, npt - npt // 3]) if isinstance(ns, tuple) else None
    n = 2 if ids is not None else 1
    kw = dict(lcids=ids, pbids=[0] * n, epids=[0] * n, nsamples=ns if n == 2 else [ns], exptimes=[0.01] * n)
    if kind == 'ma':
        m = QuadraticModel()
        args = (k[:, None], ldc, t0, p, a, inc, z, z)
    elif kind == 'ec':
        m = EclipseModel()
        args = (k, t0 - p / 2, p, a, inc, z, z)
    else:
        m = OblatePlanetModel('quadratic', nlines=20)
        args = (k[:, None], z + 0.1, z + 0.4, ldc[:, None], t0[:, None], p, a, inc, z, z)
    m.set_data(t, **kw)
    got, plain = both(m, args)
    assert np.isfinite(got).all() and got.min() < 0.999
    assert np.array_equal(got, plain)


# light curves one after another, and (apart) each with a transit of its own; the bits move
# each of these calls between the window kernel and the tile kernel
@pytest.mark.parametrize('precision,npv,npt,nlc,ns,span', [
    ('fp64', 40, 2000, 3, (1,), 2.0), ('fp64', 700, 3073, 12, (1,), 4.0),    # one sample
    ('fp64', 2100, 4097, 12, (2, 30), 0.5),                                  # uneven, many samples
    ('mixed', 40, 3000, 3, (2, 30), 0.3),                                    # a small call that fills tiles
    ('mixed', 2800, 3000, 12, (2, 30), 0.5), ('mixed', 2800, 3000, 12, (1, 5), 0.1)])
@pytest.mark.parametrize('apart', [False, True])
def test_roadrunner_routes(gpu, precision, npv, npt, nlc, ns, span, apart):
    p, a, inc, k, t0, ldc, z = orbits(npv)
    t = np.linspace(-span / 3, span, npt)
    ids = np.arange(npt) * nlc // npt
    if apart:
        t += (p[0] * np.arange(nlc))[ids]
    nss = [ns[i % len(ns)] for i in range(nlc)]
    m = RoadRunnerModel('quadratic', precision=precision)
    m.set_data(t, lcids=ids, pbids=[0] * nlc, epids=[0] * nlc, nsamples=nss, exptimes=[0.01] * nlc)
    got, plain = both(m, (k[:, None], ldc[:, None], t0[:, None], p, a, inc, z, z))
    assert np.isfinite(got).all() and got.min() < 0.999
    assert np.array_equal(got, plain)
