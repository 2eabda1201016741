"""Large copies to and from the caller's memory (16 MB and more, through
pinned pieces of 2 MB) against the same arrays moved in parts below that size:
the bytes are the same.  Totals just above the line, not a whole number of
pieces, and of many spans."""
import numpy as np
import pytest

from swfwi_amd import capi, workloads
from swfwi_amd.batch import Batch, Group
from swfwi_amd.enkf import Enkf

from test_gpu_batch import models_for

pytestmark = pytest.mark.gpu
LINE = 16 << 20


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if capi.device_count() < 1:
        pytest.skip("no HIP device")


def same(a, b):
    return np.array_equal(np.ascontiguousarray(a).view(np.uint32), np.ascontiguousarray(b).view(np.uint32))


@pytest.mark.parametrize("nt,ns", [(699, 30), (700, 30), (1501, 19)])  # 16 MB less 13 KB, and 11 KB more
def test_shots(nt, ns):
    nx, nz, nb = 200, 40, 12
    gx = np.arange(nx, dtype=np.int32)
    sx = (np.arange(ns) * 6 % nx).astype(np.int32)
    case = workloads.Case("copy", nz, nx, 10.0, nb, 0.001, nt, 20.0, sx, np.ones_like(sx), gx, np.zeros_like(gx),
                          1500.0, 3000.0, seed=3)
    vt = capi.expand_domain(workloads.models(case)[0], nb, case.dx, case.dt)
    wlt = capi.ricker(nt, case.fm, case.dt, case.amp)

    def shots(k):
        s = capi.Solver(nx, nz, nb, case.dt, case.dx, case.fm, nt, sx[k], np.ones_like(sx[k]), gx, np.zeros_like(gx))
        s.bind_velocity(vt)
        d = s.forward_shots(wlt)
        s.close()
        return d

    whole = shots(slice(None))
    print(f"shots {whole.nbytes / LINE:.4f} of the line", flush=True)
    parts = [shots(slice(k, k + 6)) for k in range(0, ns, 6)]
    assert all(p.nbytes < LINE for p in parts)
    assert np.count_nonzero(whole) > whole.size // 2
    assert same(whole, np.concatenate(parts))


def test_batch_traces():
    group = lambda k: Group(nx=150, nz=60, nb=12, dx=10.0, dt=0.001, fm=20.0, nt=801,  # noqa: E731
                            sx=np.arange(5, 145, 3)[k], sz=np.full(47, 2)[k], ng=150)
    vt, vi = models_for(group(slice(None)), 3)
    rng = np.random.default_rng(2)

    def run(k, dobs):
        b = Batch([group(k)])
        b.bind_model(0, 0, vi)
        d = b.forward()
        v = b.adjoint_source(dobs)
        g, _ = b.backward(v * np.float32(0.5))
        b.close()
        return d, v, g

    dobs = rng.standard_normal(47 * 801 * 150).astype(np.float32)
    assert dobs.nbytes > LINE
    whole = run(slice(None), dobs)
    per = 801 * 150
    parts = [run(slice(k, min(k + 16, 47)), dobs[k * per:min(k + 16, 47) * per]) for k in range(0, 47, 16)]
    for a, b in zip(whole, zip(*parts)):
        assert np.count_nonzero(a) > 0
        assert same(a, np.concatenate(b))


def test_members():
    one = np.array([3], np.int32)
    s = capi.Solver(501, 301, 12, 0.001, 10.0, 15.0, 5, one, one, one, one)
    s.bind_velocity(np.full(s.shape, 5.0, np.float32))
    e = Enkf(s, np.ones(5, np.float32), np.zeros((1, 5, 1), np.float32), 1.0, 25)
    m = np.random.default_rng(1).uniform(3, 9, (25,) + s.shape).astype(np.float32)
    assert m.nbytes > LINE
    e.set_members(m)
    assert same(e.members(), m)
    e.close()
    s.close()
