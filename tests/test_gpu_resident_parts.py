"""Batches that run as several resident launches, one after the other: the
same bits as one launch per step, also where the last part is smaller, where a
part spans two models and where the backward's parts are not the forward's."""
import numpy as np
import pytest

from swfwi_amd import capi, workloads

from test_gpu_parity import bits
from test_gpu_resident import acquisition

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if capi.device_count() < 1:
        pytest.skip("no HIP device")


@pytest.mark.parametrize("precision", [capi.PREC_EXACT, capi.PREC_FP32])
@pytest.mark.parametrize("ns,nx,nz", [(13, 301, 201), (17, 301, 201), (33, 301, 201), (5, 921, 301), (8, 921, 301),
                                      (60, 120, 90), (79, 120, 90),
                                      (39, 301, 201), (63, 301, 201)])
def test_parts_match_the_per_step_kernels(ns, nx, nz, precision):
    case = acquisition(nx, nz, 20)
    sx = np.linspace(1, nx - 2, ns).astype(np.int32)
    s = capi.Solver(nx, nz, 20, case.dt, case.dx, case.fm, case.nt, sx, np.ones_like(sx), case.gx, case.gz, precision)
    v = workloads.models(case)[0]
    wlt = capi.ricker(case.nt, case.fm, case.dt, 1.0)
    out, got = [], []
    for mode in (0, -1):
        print(f"batch of {ns} on {nx}x{nz}, resident {mode}", flush=True)
        s.set_resident(mode)
        s.bind_velocity(capi.expand_domain(v, 20, case.dx, case.dt))
        out.append(s.forward_shots(wlt))
        s.bind_velocity(capi.expand_domain(workloads.smoothed(v, 4.0), 20, case.dx, case.dt))
        inv = capi.Inversion(s, wlt, out[0], 1400.0, 3600.0, 3, 200.0)
        inv.fwi_epoch(0)
        got.append((inv.gradient(), s.velocity(), inv.stats()["obj1"], inv.stats()["obj3"]))
        inv.close()
    assert np.count_nonzero(out[0]) > 0 and np.count_nonzero(got[0][0]) > 0
    assert np.array_equal(bits(out[0]), bits(out[1]))
    assert np.array_equal(bits(got[0][0]), bits(got[1][0])) and np.array_equal(bits(got[0][1]), bits(got[1][1]))
    assert got[0][2:] == got[1][2:]
    s.close()


def test_parts_that_wait_in_vain_are_done_again_per_step():
    """No patience: whichever part gives up, the whole run is done again."""
    case = acquisition(301, 201, 20)
    sx = np.linspace(1, 299, 22).astype(np.int32)
    s = capi.Solver(301, 201, 20, case.dt, case.dx, case.fm, case.nt, sx, np.ones_like(sx), case.gx, case.gz,
                    capi.PREC_EXACT)
    s.bind_velocity(capi.expand_domain(workloads.models(case)[0], 20, case.dx, case.dt))
    wlt = capi.ricker(case.nt, case.fm, case.dt, 1.0)
    s.set_resident(0)
    want = s.forward_shots(wlt)
    for wait_us in (0.0, 5e5, 0.0):
        print(f"wait limit {wait_us} us", flush=True)
        s.set_resident(-1, wait_us)
        assert np.array_equal(bits(s.forward_shots(wlt)), bits(want))
    s.close()
