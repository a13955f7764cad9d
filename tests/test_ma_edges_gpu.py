"""The Mandel-Agol model outside its usual parameters: negative radius ratios, which a
sampler without bounds proposes and which give NaN under the disk as the reference's
square root of a negative modulus does; coefficients whose disk integral is 0; planets
as large as the star and larger, against the FP64 oracle (1e-9 absolute, the suite's bar)."""
import numpy as np
import pytest

from pytransit_amd import QuadraticModel

pytestmark = pytest.mark.gpu

P, A, I = 3.2, 9.5, 1.55
LAYOUTS = [dict(), dict(nsamples=3, exptimes=0.01), dict(lcids=np.repeat([0, 1], [150, 151]), nsamples=[1, 2], exptimes=[0.0, 0.01])]


def evaluate(t, k, ldc, **data):
    tm = QuadraticModel()
    tm.set_data(t, **data)
    n = len(k)
    return np.atleast_2d(tm.evaluate(np.reshape(k, (n, 1)), np.asarray(ldc, float), np.full(n, 0.001), np.full(n, P),
                                     np.full(n, A), np.full(n, I)))


def separations(oracle, t, data):
    """Smallest and largest separation of each exposure's samples; the window's points."""
    lc = np.asarray(data.get('lcids', np.zeros(t.size, int)))
    ns = np.broadcast_to(data.get('nsamples', 1), lc.max() + 1)[lc]
    ex = np.broadcast_to(data.get('exptimes', 0.0), lc.max() + 1)[lc]
    c = oracle.taylor_coeffs(P, A, I, 0.0, 0.0)
    return [np.array([oracle.sep(x - 0.001 + e * ((s - 0.5) / n - 0.5), c) for s in range(1, n + 1)])
            for x, n, e in zip(t, ns, ex)]


@pytest.mark.parametrize('data', LAYOUTS)
def test_negative_radius_ratio(gpu, oracle, data):
    t = np.linspace(-0.1, 0.1, 301)
    k = np.array([-0.1, 0.1, -1e-4, -0.9, -1.5])
    f = evaluate(t, k, np.tile([0.3, 0.2], (5, 1)), **data)
    z = separations(oracle, t, data)
    for i in (0, 2, 3, 4):
        low = np.array([v.min() for v in z])
        clear = np.abs(low - (1.0 + k[i])) > 1e-6
        under = low <= 1.0 + k[i]
        window = np.abs(t - 0.001) < 0.04              # inside the contacts of every k here
        assert np.isnan(f[i][under & clear & window]).all()
        assert (f[i][~under & clear] == 1.0).all()
    assert (under & clear & window).sum() == 0 and np.isnan(f[0]).any()
    assert np.isfinite(f[1]).all() and f[1].min() < 0.99


# (one sample an exposure: infinities of both signs in one exposure have no mean)
@pytest.mark.parametrize('data', [dict(), dict(lcids=np.repeat([0, 1], [150, 151]))])
def test_vanishing_disk_integral(gpu, data):
    """1 - u1/3 - u2/6 = 0 exactly: infinities, as an IEEE quotient by 0 gives."""
    t = np.linspace(-0.1, 0.1, 301)
    f = evaluate(t, [0.1, 0.1], [[1.5, 3.0], [0.3, 0.2]], **data)
    assert not np.isnan(f).any()
    assert np.isinf(f[0]).sum() > 100 and ((f[0] == 1.0) | np.isinf(f[0])).all()
    assert np.isfinite(f[1]).all()


@pytest.mark.parametrize('data', LAYOUTS)
def test_large_planets(gpu, oracle, data):
    t = np.linspace(-0.25, 0.25, 301)
    k = np.array([0.49995, 0.5, 0.9, 1.0, 1.2, 3.0])
    ldc = np.tile([0.35, 0.2], (6, 1))
    f = evaluate(t, k, ldc, **data)
    nlc = int(np.max(data.get('lcids', 0))) + 1
    full = lambda x, dt: np.broadcast_to(np.asarray(x, dt), nlc)
    ref = oracle.quadratic_model(t, k[:, None], np.full((6, 1), 0.001), np.full(6, P), np.full(6, A), np.full(6, I),
                                 np.zeros(6), np.zeros(6), np.tile(ldc, (1, 1)), data.get('lcids', np.zeros(301, int)),
                                 np.zeros(nlc, int), np.zeros(nlc, int), full(data.get('nsamples', 1), int),
                                 full(data.get('exptimes', 0.0), float))
    assert ref.min() == 0.0 and np.isfinite(ref).all()
    assert np.abs(f - ref).max() <= 1e-9
