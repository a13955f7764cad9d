"""Which inputs of the likelihood are read where they are: numbers and float64 tensors on the
device with one value or one per vector.  Everything else takes the general path, which
copies or refuses it."""
import numpy as np
import pytest
import torch

from pytransit_amd.rrmodel import RoadRunnerModel, _vec_in_place

CPU = torch.device('cpu')


def f64(*shape):
    return torch.arange(1.0, 1.0 + int(np.prod(shape)), dtype=torch.float64).reshape(shape)


def test_read_in_place():
    base = f64(4, 3)
    for x, stride in ((base[:, 1], 3), (base[:, 1:2], 3), (f64(4), 1), (f64(1).expand(4), 0), (f64(1), 0), (f64(1, 1), 0),
                      (torch.tensor(2.0, dtype=torch.float64), 0)):
        v = _vec_in_place(x, 4, CPU)
        assert v.ptr == x.data_ptr() and v.stride == stride
    assert _vec_in_place(2, 4, CPU).value == 2.0 and _vec_in_place(np.float64(0.5), 4, CPU).value == 0.5


@pytest.mark.parametrize('x', [f64(3), f64(2, 2), f64(1, 4), f64(1, 1, 1), f64(4, 1, 1), f64(4).float(), np.ones(4), [1.0], None,
                               torch.complex(f64(4), f64(4)).conj().imag, torch.complex(f64(1), f64(1)).conj().imag])
def test_not_read_in_place(x):
    assert _vec_in_place(x, 4, CPU) is None


def test_radius_ratios_of_three_dimensions_are_refused():
    """As in evaluate; a single value in three dimensions was read in place."""
    m = RoadRunnerModel('quadratic', device='cpu')
    with pytest.raises(Exception):
        m._params(f64(1, 1, 1), f64(4), f64(4), f64(4), f64(4), 0.0, 0.0, CPU)
