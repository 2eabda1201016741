"""Forward batches whose resident tiles run two blocks a CU: 1 to 6 rows a
wave, ragged last columns, against one launch per step, bit for bit."""
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
@pytest.mark.parametrize("ns,nx,nz", [(1, 700, 200), (2, 301, 201), (5, 301, 201), (8, 301, 201), (11, 299, 203),
                                      (13, 301, 201), (16, 301, 201), (2, 921, 301), (4, 921, 301)])
def test_two_blocks_a_cu(ns, nx, nz, precision):
    case = acquisition(nx, nz, 20)
    sx = np.linspace(1, nx - 2, ns).astype(np.int32)
    s = capi.Solver(nx, nz, 20, case.dt, case.dx, case.fm, case.nt, sx, np.ones_like(sx), case.gx, case.gz, precision)
    s.bind_velocity(capi.expand_domain(workloads.models(case)[0], 20, case.dx, case.dt))
    wlt = capi.ricker(case.nt, case.fm, case.dt, 1.0)
    out = []
    for mode in (0, 1):
        print(f"batch of {ns} on {nx}x{nz}, resident {mode}", flush=True)
        s.set_resident(mode)
        out.append(s.forward_shots(wlt))
    assert np.count_nonzero(out[0]) > 0
    assert np.array_equal(bits(out[0]), bits(out[1]))
    s.close()
