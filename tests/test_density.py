"""The density bits of a data set: floor(log2) of the times in a tenth of a day and of the
mean number of samples, unset where the density is below 16 or cannot be told."""
import warnings

import numpy as np
import pytest

from pytransit_amd import transitmodel

one = lambda n: np.ones(n, int)


def density_bits(t, ns):
    """Every point in a light curve of its own."""
    return transitmodel.density_bits(t, np.arange(t.size), ns)


def parts(bits):
    assert bits & 0xff == 0 and bits >> 18 == 0
    return bits >> 8 & 31, bits >> 13


@pytest.mark.parametrize('npt', [65, 1000, 1026, 5000])
@pytest.mark.parametrize('per', [17.0, 63.0, 65.0, 900.0, 1e6])
def test_even_steps(npt, per):
    t = 2459000.0 * (per < 1e5) + np.arange(npt) * 0.1 / per
    assert parts(density_bits(t, one(npt))) == (int(np.log2(per)), 0)
    assert parts(density_bits(t[::-1].copy(), 5 * one(npt))) == (int(np.log2(per)), 2)


def test_gaps_and_shared_times():
    night = np.arange(400) * 1e-3                      # 100 times in a tenth of a day
    t = (night + 30 * np.arange(12)[:, None]).ravel()
    assert parts(density_bits(t, one(t.size)))[0] == 6
    t = np.repeat(np.arange(800) * 1e-3, 2)            # two light curves at the same times: twice as many
    assert parts(density_bits(t, one(t.size)))[0] == 7


def test_unknown():
    rng = np.random.default_rng(0)
    assert density_bits(np.arange(5000) * 0.1 / 15.0, one(5000)) == 0
    assert density_bits(np.arange(64) * 1e-4, one(64)) == 0
    assert density_bits(rng.permutation(np.linspace(0, 30, 5000)), one(5000)) == 0
    with warnings.catch_warnings():
        warnings.simplefilter('error')
        for t in (np.full(500, np.nan), np.full(500, np.inf), np.zeros(500), np.zeros(0)):
            assert density_bits(t, one(t.size)) == 0
    assert transitmodel.density_bits(np.arange(500) * 1e-3, np.zeros(500, int), np.array([6])) == 6 << 8 | 2 << 13


def test_limits_of_the_fields():
    t = np.arange(200) * 5e-324
    assert parts(density_bits(t, one(200))) == (30, 0)
    t = np.arange(200) * 1e-300
    assert parts(density_bits(t, np.full(200, 2 ** 40))) == (30, 30)
    assert parts(density_bits(np.arange(200) * 1e-3, np.repeat([2, 30], 100)))[1] == 4
