"""Copies of a model (``copy.deepcopy``, ``pickle``) have device arrays of their own: the
addresses that go to the kernels are the copy's, and stay valid when the original gets
other data.  On CPU tensors, which have addresses too."""
import copy
import pickle

import numpy as np
import pytest
import torch

from pytransit_amd import EclipseModel, EclipseSpectroscopyModel, QuadraticModel

CPU = torch.device('cpu')
FIELDS = ('times', 'lcids', 'pbids', 'epids', 'nsamples', 'exptimes')


def addresses(model, epids='epids'):
    lc = model._lc_descriptor(CPU, model.npb, 1, epids)
    return [getattr(lc, f) for f in FIELDS]


def own(model, epids='epids'):
    d = model._device_data(CPU)
    return [d[epids if f == 'epids' else f].data_ptr() for f in FIELDS]


@pytest.mark.parametrize('cls', [QuadraticModel, EclipseModel, EclipseSpectroscopyModel])
@pytest.mark.parametrize('dup', [copy.deepcopy, copy.copy, lambda m: pickle.loads(pickle.dumps(m))])
@pytest.mark.parametrize('epids', ['epids', 'pbids'])
def test_a_copy_reads_its_own_arrays(cls, dup, epids):
    m = cls()
    m.set_data(np.linspace(-0.1, 0.1, 50), lcids=np.repeat([0, 1], 25), nsamples=[1, 3], exptimes=[0.0, 0.01])
    assert addresses(m, epids) == own(m, epids)
    c = dup(m)
    assert addresses(c, epids) == own(c, epids)
    m.set_data(np.linspace(-0.2, 0.2, 70))
    assert addresses(m, epids) == own(m, epids) and addresses(c, epids) == own(c, epids)
    assert c.npt == 50 and c._lc_descriptor(CPU, 1, 1).npt == 50
