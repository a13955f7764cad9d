"""A separation whose square overflows is off the disk: the spectroscopy models' flux is
exactly 1 there, as in the FP64 oracle, in every form of the flux kernel."""
import numpy as np
import pytest

from pytransit_amd import TSModel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('precision', ['fp64', 'mixed'])
@pytest.mark.parametrize('npv,npb,npt,nss', [(3, 2, 301, 1), (3, 2, 301, 3), (3, 2, 70, 40), (300, 40, 2500, 1)])
def test_far_orbit(gpu, oracle, precision, npv, npb, npt, nss):
    t = np.linspace(-0.2, 0.2, npt)
    ext = 0.01 if nss > 1 else 0.0
    tm = TSModel('quadratic', precision=precision)
    tm.set_data(t, nsamples=nss, exptimes=ext)
    k = np.full((npv, npb), 0.1)
    ldc = np.full((npv, npb, 2), 0.2)
    a = np.full(npv, 1e200)
    a[1] = 9.0
    full = lambda x: np.full(npv, float(x))
    f = tm.evaluate(k, ldc, full(0.001), full(3.0), a, full(1.55))
    ze, _ = oracle.create_z_grid(0.7, 20, 20)
    ldp, istar = oracle.evaluate_ld('quadratic', tm.mu, ldc[:1])
    with np.errstate(over='ignore'):
        ref = oracle.tsmodel_serial(t, k[:1], full(0.001)[:1], full(3.0)[:1], a[:1], full(1.55)[:1], full(0)[:1], full(0)[:1], nss,
                                    ext, ldp, istar, None, 0, 0, 0, 100, 0, ze)
    assert (ref == 1.0).all()
    assert (np.delete(f, 1, 0) == 1.0).all() and f[1].min() < 0.995
