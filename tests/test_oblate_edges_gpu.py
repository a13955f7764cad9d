"""The oblate planet at the ends of its ranges against the FP64 oracle (1e-9 absolute):
flattenings past 1, whose chords have swapped ends; the most scanlines (49 KB of LDS,
beside up to 43 KB for the points) for one and several light curves and for one and
four times a lane; the last number of scanlines accepted."""
import numpy as np
import pytest

from oracle import ec_oracle
from pytransit_amd import OblatePlanetModel

pytestmark = pytest.mark.gpu


def both(oracle, t, f, alpha, nlines, rows=None, lcids=None, nsamples=(2,), exptimes=(0.005,), k=None):
    n = len(f)
    rows = np.arange(n) if rows is None else rows
    k = np.linspace(0.08, 0.2, n) if k is None else k
    ldc = np.tile([0.4, 0.2], (n, 1))[:, None, :]
    full = lambda x: np.full(n, float(x))
    # inclinations from central to grazing transits
    args = (full(0.001)[:, None], full(3.0), full(9.0), np.linspace(1.47, 1.56, n), full(0.0), full(0.0))
    m = OblatePlanetModel('quadratic', nlines=nlines)
    nlc = len(nsamples)
    m.set_data(t, lcids=lcids, pbids=[0] * nlc, nsamples=nsamples, exptimes=exptimes)
    got = np.atleast_2d(m.evaluate(k[:, None], f, alpha, ldc, *args))
    orr = oracle.OracleRR('quadratic')
    ldp, istar = orr.ld(ldc[rows])
    ids = np.zeros(t.size, int) if lcids is None else lcids
    ref = ec_oracle.opmodel(t, k[rows][:, None], f[rows], alpha[rows], *(x[rows] for x in args), nlc, 1, 1, nlines, ids,
                            np.zeros(nlc, int), np.zeros(nlc, int), np.array(nsamples), np.array(exptimes, float), ldp, istar,
                            orr.weights, orr.dk, 0.005, 0.5, orr.dg, orr.ze)
    return got[rows], np.atleast_2d(ref)


def test_flattening_past_one(gpu, oracle):
    f = np.array([1.5, 1.2, 3.0, 0.3, 0.999, -0.4])
    got, ref = both(oracle, np.linspace(-0.12, 0.12, 301), f, np.array([0.3, -1.1, 2.0, 0.0, 1.5, 0.7]), 60)
    assert ref.max() > 1 + 1e-4 and ref.min() < 0.99
    assert np.abs(got - ref).max() <= 1e-9


# npv and npt: one time a lane; four, in several sub-tiles a workgroup (checked on three vectors)
@pytest.mark.parametrize('npv,npt', [(3, 301), (1100, 8200)])
@pytest.mark.parametrize('lcs', [False, True])
def test_most_scanlines(gpu, oracle, npv, npt, lcs):
    rng = np.random.default_rng(npv)
    # the transit in the first few hundred points: the oracle's time goes with the points in the window
    t = np.concatenate([np.linspace(-0.1, 0.1, 240), np.linspace(0.1, 1.4, npt - 240)])
    kw = dict(lcids=np.repeat([0, 1], [100, npt - 100]), nsamples=(1, 2), exptimes=(0.0, 0.005)) if lcs else {}
    rows = np.array([0, npv // 2, npv - 1])
    got, ref = both(oracle, t, rng.uniform(0.0, 0.4, npv), rng.uniform(-2, 2, npv), 2048, rows, **kw)
    assert ref.min() < 0.99
    assert np.abs(got - ref).max() <= 1e-9


def test_too_many_scanlines_are_refused(gpu):
    m = OblatePlanetModel('quadratic', nlines=2049)
    m.set_data(np.linspace(-0.1, 0.1, 11))
    with pytest.raises(Exception, match='nlines'):
        m.evaluate(0.1, 0.1, 0.0, [0.4, 0.2], 0.0, 3.0, 9.0, 1.55)


# the number of lanes that share a sample's scanlines changes at 16, 48 and 128 lines, and
# at four samples a point
@pytest.mark.parametrize('nlines', [2, 15, 16, 47, 48, 65, 127, 128])
@pytest.mark.parametrize('ns', [1, 3, 4, (1, 6)])
def test_lanes_of_a_sample(gpu, oracle, nlines, ns):
    t = np.linspace(-0.12, 0.12, 301)
    kw = dict(lcids=np.repeat([0, 1], [130, 171]), nsamples=ns, exptimes=(0.0, 0.01)) if ns == (1, 6) else \
        dict(nsamples=(ns,), exptimes=(0.01,))
    got, ref = both(oracle, t, np.array([0.0, 0.2, 1.3]), np.array([0.1, -1.0, 2.0]), nlines, **kw)
    assert ref.min() < 0.995
    assert np.abs(got - ref).max() <= 1e-9
