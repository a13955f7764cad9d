"""Limb-darkening means from a law's basis table against the contraction of the whole
profile, for every law that has one, one and several passbands (also more than a
group), even and odd numbers of g, and a radius ratio outside the weight table."""
import numpy as np
import pytest
import torch

from pytransit_amd import RoadRunnerModel, _lib

LAWS = {'uniform': 0, 'linear': 1, 'quadratic': 2, 'quadratic-tri': 2, 'nonlinear': 4, 'square_root': 2,
        'logarithmic': 2, 'exponential': 2}

# Both forms sum the same at most 40 products of weights (which add up to 1) and
# basis values below 2 with coefficients below 1, in another order: a limb-darkening
# mean differs by at most 40 eps * 2 * 5 = 9e-14 and the flux by k^2 = 0.04 of that.
# FP32 adds the rounding of the table, the means and the flux: 3 * 6e-8.
TOL = {'fp64': 1e-14, 'mixed': 2e-7}


@pytest.mark.gpu
@pytest.mark.parametrize('precision', ['fp64', 'mixed'])
@pytest.mark.parametrize('npb, ng', [(1, 100), (3, 51), (7, 100), (70, 100)])
@pytest.mark.parametrize('law', list(LAWS))
def test_basis_table_equals_profile(law, npb, ng, precision):
    rng = np.random.default_rng(npb * ng)
    npv = 9
    time = np.tile(np.linspace(-0.1, 0.1, 40), npb)
    tm = RoadRunnerModel(law, ng=ng, klims=(0.01, 0.2), precision=precision)
    tm.set_data(time, lcids=np.repeat(np.arange(npb), 40), pbids=np.arange(npb))
    k = rng.uniform(0.05, 0.19, (npv, 1))
    k[4] = 0.25                                     # the exact weights
    ldc = rng.uniform(0.1, 0.3, (npv, npb, max(LAWS[law], 1)))
    ldc[7, 0, 0] = np.nan if LAWS[law] else 0.2
    args = (k, ldc, rng.normal(0, 1e-3, npv), rng.uniform(2, 4, npv), rng.uniform(6, 9, npv), rng.uniform(1.5, 1.57, npv))
    got = np.atleast_2d(tm.evaluate(*args)).astype(float)
    keep = tm._table(tm.device)[1]
    assert keep['basis'] is not None
    keep['basis'] = None
    want = np.atleast_2d(tm.evaluate(*args)).astype(float)
    # at the limb the trapezoid takes log(0) and 1 / (1 - exp(0)), as the reference's: these
    # two laws' disk integrals are NaN and infinite, the flux in transit NaN and 1
    assert (want < 0.999).any() or law in ('logarithmic', 'exponential')
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.nanmax(np.abs(got - want)) <= TOL[precision]


@pytest.mark.parametrize('law', [5, 9, 10, -1, 11, 0x100])
def test_laws_without_a_basis_are_refused(law):
    lib = _lib.load(require_gpu=False)
    assert lib.rr_ld_basis_count(law) == 0
    assert lib.rr_ld_basis_table(law, None, None, None) != 0
