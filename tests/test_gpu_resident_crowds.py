"""Many sources or receivers on few places of a resident tile: the amplitudes of
a place add in id order, as one launch per step does, and a step stays the faster
one of the two."""
import numpy as np
import pytest

from swfwi_amd import capi, workloads

from test_gpu_parity import bits

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if capi.device_count() < 1:
        pytest.skip("no HIP device")


def solver(nx, nz, nb, sx, sz, gx, gz, nt, precision=capi.PREC_EXACT):
    case = workloads.Case("crowd", nz, nx, 20.0, nb, 0.002, nt, 12.0, sx, sz, gx, gz, 1500.0, 3500.0, seed=nx)
    s = capi.Solver(nx, nz, nb, case.dt, case.dx, case.fm, nt, sx, sz, gx, gz, precision)
    s.bind_velocity(capi.expand_domain(workloads.models(case)[0], nb, case.dx, case.dt))
    return s, capi.ricker(nt, case.fm, case.dt, 1.0)


def times(s, run):
    """Best forward and backward microseconds a step of five runs."""
    t = []
    for _ in range(5):
        s.set_timing(True)
        run()
        t.append([1e3 * ms / n for ms, n in s.kernel_times().values()])
        s.set_timing(False)
    return np.min(t, 0)


@pytest.mark.parametrize("precision", [capi.PREC_EXACT, capi.PREC_FP32])
@pytest.mark.parametrize("nx,nz,nb,n,places", [(301, 201, 20, 480, 12), (301, 201, 20, 512, 1), (921, 301, 30, 60, 12),
                                               (921, 301, 30, 300, 299)])
def test_crowded_sources(nx, nz, nb, n, places, precision):
    i = np.arange(n)
    sx, sz = (nx // 2 + i * 7 % places % 6).astype(np.int32), (1 + i * 7 % places // 6).astype(np.int32)
    gx = np.concatenate([np.arange(0, nx, 2), [5, 5, 5]]).astype(np.int32)
    s, wlt = solver(nx, nz, nb, sx, sz, gx, np.zeros_like(gx), 180, precision)
    r = np.random.default_rng(n)
    enc = np.ascontiguousarray(wlt[:, None] * r.uniform(-1, 1, n)[None]).astype(np.float32)
    vsrc = r.standard_normal((180, gx.size)).astype(np.float32)
    got, t = [], []
    for mode in (0, -1):
        s.set_resident(mode)
        print(f"{n} sources on {places} places of {nx}x{nz}, resident {mode}", flush=True)
        got.append((s.forward_modeling(enc), s.calgradient(enc, vsrc)))
        t.append(times(s, lambda: s.calgradient(enc, vsrc)))
        assert {s.last_run(0)[0], s.last_run(1)[0]} == {"per step" if mode == 0 else "resident"}
    for a, b in zip(*got):
        assert np.count_nonzero(a) > 0 and np.array_equal(bits(a), bits(b))
    print("  microseconds a step, forward and backward:", t[0], t[1], flush=True)
    assert (t[1] < t[0]).all()
    s.close()


@pytest.mark.parametrize("nx,nz,nb,extra", [(1501, 501, 30, 60), (921, 301, 30, 60)])
def test_receivers_with_some_doubled(nx, nz, nb, extra):
    gx = np.concatenate([np.arange(nx), np.linspace(0, nx - 1, extra)]).astype(np.int32)
    one = np.array([nx // 2], np.int32)
    s, wlt = solver(nx, nz, nb, one, one * 0 + 1, gx, np.zeros_like(gx), 180)
    vsrc = np.random.default_rng(1).standard_normal((180, gx.size)).astype(np.float32)
    got, t = [], []
    for mode in (0, -1):
        s.set_resident(mode)
        print(f"{gx.size} receivers on {nx}x{nz}, resident {mode}", flush=True)
        got.append(s.calgradient(wlt, vsrc, shot=0))
        t.append(times(s, lambda: s.calgradient(wlt, vsrc, shot=0)))
        assert s.last_run(1)[0] == ("per step" if mode == 0 else "resident")
    assert np.count_nonzero(got[0]) > 0 and np.array_equal(bits(got[0]), bits(got[1]))
    print("  microseconds a step, forward and backward:", t[0], t[1], flush=True)
    assert (t[1] < t[0]).all()
    s.close()
