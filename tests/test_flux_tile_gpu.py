"""The flux kernel's tile length follows the size of the launch (128 to 1024 times): a
pv's light curve is the same to the last bit in a launch of few pvs and of thousands,
for a sorted and an unsorted light curve, times that end inside a tile, and several
light curves with one and with different numbers of samples."""
import numpy as np
import pytest

from pytransit_amd import RoadRunnerModel


@pytest.mark.gpu
@pytest.mark.parametrize('precision', ['fp64', 'mixed'])
@pytest.mark.parametrize('ns', [1, 7])
@pytest.mark.parametrize('layout, npt', [('one', 2065), ('unsorted', 2065), ('three', 2064), ('one', 130)])
def test_same_bits_for_every_tile_length(layout, npt, ns, precision):
    rng = np.random.default_rng(npt + ns)
    few, many = 5, 12000 if npt < 200 else 4000
    time = np.linspace(-0.4, 2.4, npt)
    tm = RoadRunnerModel('quadratic', precision=precision)
    if layout == 'unsorted':
        time = rng.permutation(time)
    if layout == 'three':
        tm.set_data(time, lcids=np.repeat(np.arange(3), npt // 3), pbids=np.zeros(3, int), nsamples=np.full(3, ns),
                    exptimes=np.array([0.01, 0.02, 0.01]))
    else:
        tm.set_data(time, nsamples=ns, exptimes=0.02)
    par = dict(k=rng.uniform(0.05, 0.15, few), t0=rng.normal(0, 0.01, few), p=rng.uniform(0.9, 1.6, few),
               a=rng.uniform(4, 6, few), i=rng.uniform(1.45, 1.57, few))
    ldc = rng.uniform(0.1, 0.4, (few, 1, 2))
    idx = np.arange(many) % few
    want = tm.evaluate(par['k'][:, None], ldc, par['t0'], par['p'], par['a'], par['i'])
    got = tm.evaluate(par['k'][idx, None], ldc[idx], par['t0'][idx], par['p'][idx], par['a'][idx], par['i'][idx])
    assert (want < 0.999).any()
    assert np.array_equal(got, want[idx])
