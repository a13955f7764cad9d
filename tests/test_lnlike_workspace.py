"""The likelihood's workspace: what a precision and the gradient need, and a bound for any
number of parameter vectors, which are then taken in parts."""
import numpy as np
import pytest
import torch

from pytransit_amd import RoadRunnerModel, _lib


def size(prec, grad, npv, npt=1000, ng=100):
    return _lib.load(require_gpu=False).rr_lnlike_vec_workspace_bytes(prec, grad, npv, npt, ng)


def test_workspace_is_bounded():
    for prec in (_lib.RR_FP64, _lib.RR_MIXED):
        for grad in (0, 1):
            assert max(size(prec, grad, n) for n in (32768, 32769, 65537, 10 ** 6, 2 ** 31 - 1)) < 256 << 20
            assert size(prec, grad, 1000) < size(prec, grad, 2000) < size(prec, grad, 32768)
    # a record of 256 bytes, 100 FP32 values, the vector's sums
    assert size(_lib.RR_MIXED, 0, 30000) < 30000 * (256 + 400 + 64) + 65536
    # a workspace of the precision-free size serves every form
    lib = _lib.load(require_gpu=False)
    for npv in (0, 1, 7, 5000, 40000, 10 ** 6):
        most = lib.rr_lnlike_workspace_bytes(npv, 1000, 100)
        assert all(size(prec, grad, npv) <= most for prec in (_lib.RR_FP64, _lib.RR_MIXED) for grad in (0, 1))


@pytest.mark.gpu
@pytest.mark.parametrize('precision', ['fp64', 'mixed'])
def test_parts_give_the_same_bits(gpu, precision):
    """Vectors on both sides of a part's end, and the last, as on their own."""
    npv, rng = 65537, np.random.default_rng(4)
    t = np.linspace(-0.1, 0.1, 60)
    m = RoadRunnerModel('quadratic', precision=precision)
    m.set_data(t, nsamples=2, exptimes=0.01)
    th = np.column_stack([rng.uniform(0.05, 0.15, npv), rng.normal(0, 1e-3, npv), rng.uniform(2, 4, npv),
                          rng.uniform(8, 12, npv), rng.uniform(1.5, 1.57, npv), rng.uniform(0.1, 0.4, (npv, 2))])
    obs, sigma = np.where(np.abs(t) < 0.05, 0.99, 1.0), rng.uniform(2e-4, 4e-4, npv)
    th = torch.as_tensor(th, device=gpu)
    sg = torch.as_tensor(sigma, device=gpu)

    def call(rows, grad):
        x, s = th[rows], sg[rows]
        return m.lnlike(x[:, 0], x[:, None, 5:7], x[:, 1], x[:, 2], x[:, 3], x[:, 4], obs, s, grad=grad)
    lnl, g = call(slice(None), True)
    plain = call(slice(None), False)
    assert np.isfinite(lnl).all() and np.isfinite(g).all()
    chunk = -(-npv // 3)
    for rows in (slice(0, 5), slice(chunk - 3, chunk + 3), slice(2 * chunk - 2, 2 * chunk + 2), slice(npv - 4, npv)):
        l1, g1 = call(rows, True)
        assert np.array_equal(l1, lnl[rows]) and np.array_equal(g1, g[rows])
        assert np.array_equal(call(rows, False), plain[rows])
