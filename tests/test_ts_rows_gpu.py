"""The forms of the spectroscopy flux that write whole rows: the plain FP32 form on the grids
that the aligned form does not take (129 to 249 g) against the FP64 oracle (1 ppm), and the
space around the flux of every row form, untouched."""
import numpy as np
import pytest
import torch

from pytransit_amd import TabulatedLDModel, TSModel, _lib, workloads

pytestmark = pytest.mark.gpu

MU = dict(nzin=24, nzlimb=24)


def workload(npv, npb, npt, ng, seed):
    return workloads.ts_many_pb(npv=npv, npt=npt, npb=npb, seed=seed, mu=TSModel('quadratic', **MU).mu)


def reference(oracle, wl, r, ng):
    ze, _ = oracle.create_z_grid(0.7, 24, 24)
    return oracle.tsmodel_serial(wl.times, wl.k[r], wl.t0[r], wl.p[r], wl.a[r], wl.i[r], wl.e[r], wl.w[r], 1, 0.0, wl.ldp[r],
                                 wl.istar[r], None, 0, 0, 0, ng, 0, ze)


# from 24 million values: both ends of the grids, one passband past a workgroup's and one short,
# the longest rows
@pytest.mark.parametrize('npv,npb,npt,ng', [(270, 33, 2704, 129), (270, 31, 2900, 249), (90, 97, 8192, 200)])
def test_plain_fp32_rows(gpu, oracle, npv, npb, npt, ng):
    assert npv * npb * npt >= 24000000
    wl = workload(npv, npb, npt, ng, npt)
    wl.a[1] = 0.5                           # an invalid vector
    tm = TSModel(TabulatedLDModel(wl.ldp, wl.istar), ng=ng, precision='mixed', **MU)
    tm.set_data(wl.times)
    f = tm.evaluate(wl.k, None, wl.t0, wl.p, wl.a, wl.i)
    assert np.isnan(f[1]).all() and not np.isnan(np.delete(f, 1, 0)).any()
    r = np.array([0, 1, npv // 2, npv - 1])
    ref = reference(oracle, wl, r, ng)
    assert np.nanmin(ref) < 1
    assert np.nanmax(np.abs(f[r] - ref)) <= 1e-6


# the aligned form from a cache line's row on, with heads of 0 to 7 vectors; the plain forms; the tiles
@pytest.mark.parametrize('precision,npv,npb,npt,ng', [
    ('mixed', 257, 3, 4, 100), ('mixed', 256, 9, 20, 100), ('mixed', 256, 6, 32, 100), ('mixed', 260, 3, 36, 100),
    ('mixed', 130, 33, 2052, 100), ('mixed', 70, 65, 8192, 100), ('mixed', 300, 40, 2004, 129), ('mixed', 5, 33, 1237, 100),
    ('fp64', 260, 33, 3000, 100), ('fp64', 300, 31, 2600, 100), ('fp64', 3, 17, 65, 100)])
def test_nothing_outside_the_flux_is_written(gpu, oracle, precision, npv, npb, npt, ng, monkeypatch):
    wl = workload(npv, npb, npt, ng, npt)
    tm = TSModel(TabulatedLDModel(wl.ldp, wl.istar), ng=ng, precision=precision, **MU)
    tm.set_data(wl.times)
    ref = tm.evaluate(wl.k, None, wl.t0, wl.p, wl.a, wl.i)
    dtype = torch.float32 if precision == 'mixed' else torch.float64
    n, guard = npv * npb * npt, 1024
    buffer = torch.full((n + 2 * guard,), -3.0, dtype=dtype, device=gpu)
    real = torch.empty

    def empty(shape, **kw):
        return buffer[guard:guard + n].view(shape) if tuple(np.atleast_1d(shape)) == (npv, npb, npt) else real(shape, **kw)
    monkeypatch.setattr(torch, 'empty', empty)
    f = tm.evaluate(wl.k, None, wl.t0, wl.p, wl.a, wl.i, copy=False)
    monkeypatch.undo()
    assert f.data_ptr() == buffer[guard:].data_ptr()
    b = buffer.cpu().numpy()
    assert (b[:guard] == -3.0).all() and (b[guard + n:] == -3.0).all()
    assert np.array_equal(b[guard:guard + n].reshape(ref.shape), ref, equal_nan=True)
