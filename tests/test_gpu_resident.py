"""The resident time loop (one launch per run, tiles kept on the chip) against
the CPU oracle: bit-identical in exact mode, whatever the tile edges."""
import numpy as np
import pytest

from swfwi_amd import capi, workloads

from test_gpu_parity import bits, setup_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if capi.device_count() < 1:
        pytest.skip("no HIP device")


def acquisition(nx, nz, nb, nt=180):
    """Sources and receivers on and beside tile edges, some of them coincident;
    dt = 2 ms, so that the imaging condition starts at step 151."""
    sx = np.array([0, nx // 2, nx // 2, nx - 1], np.int32)
    sz = np.array([1, nz - 1, nz - 1, nz // 2], np.int32)
    gx = np.concatenate([np.arange(nx), [3, 3]]).astype(np.int32)
    gz = np.concatenate([np.zeros(nx), [nz - 1, nz - 1]]).astype(np.int32)
    return workloads.Case("edges", nz, nx, 20.0, nb, 0.002, nt, 12.0, sx, sz, gx, gz, 1500.0, 3500.0, seed=nx + nz)


# update region (nx + 2 nb) x (nz + nb): z around one and two tiles of 62, x
# around one, two and many tiles of 8 and one row more; then wider tiles (a
# model of 501 x 1501 has 56), odd and even step counts
@pytest.mark.parametrize("nx,nz,nb,nt", [(4, 56, 6, 180), (5, 57, 6, 181), (21, 118, 6, 180), (20, 119, 6, 181),
                                         (333, 201, 20, 180), (301, 61, 7, 181), (921, 301, 30, 160),
                                         (1501, 501, 30, 158)])
def test_edges_bitexact(oracle, nx, nz, nb, nt):
    case = acquisition(nx, nz, nb, nt)
    s, g, vt, vi, wlt = setup_case(oracle, case)
    s.set_resident(1)
    s.bind_velocity(vt)
    enc = oracle.encode_source(capi.random_codes(3, case.ns), wlt) * np.float32(1.37)
    vsrc = np.random.default_rng(nt).standard_normal((case.nt, case.ng)).astype(np.float32)
    print(f"resident {nx}x{nz} nb={nb} nt={nt}", flush=True)
    assert np.array_equal(bits(s.forward_modeling(enc)), bits(g.forward_modeling(vt, enc, shot=-1)))
    assert np.array_equal(bits(s.forward_modeling(wlt, shot=1)), bits(g.forward_modeling(vt, wlt, shot=1)))
    assert np.array_equal(bits(s.calgradient(enc, vsrc)), bits(g.calgradient(vt, enc, vsrc, shot=-1)))
    assert np.array_equal(bits(s.calgradient(wlt, vsrc, shot=3)), bits(g.calgradient(vt, wlt, vsrc, shot=3)))


@pytest.mark.parametrize("precision", [capi.PREC_EXACT, capi.PREC_FP32])
@pytest.mark.parametrize("ns,nx,nz", [(2, 150, 90), (7, 201, 130), (13, 301, 201), (21, 301, 201)])
def test_batches_match_the_per_step_kernels(ns, nx, nz, precision):
    """Several entries in one launch, every tile width that takes: the same
    bits as one launch per step."""
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
    assert np.array_equal(bits(out[0]), bits(out[1]))
    v0 = workloads.smoothed(workloads.models(case)[0], 4.0)
    got = []
    for mode in (0, 1):
        s.set_resident(mode)
        s.bind_velocity(capi.expand_domain(v0, 20, case.dx, case.dt))
        inv = capi.Inversion(s, wlt, out[0], 1400.0, 3600.0, 3, 200.0)
        inv.fwi_epoch(0)
        got.append((inv.gradient(), s.velocity(), inv.stats()["obj1"], inv.stats()["obj3"]))
        inv.close()
    assert np.array_equal(bits(got[0][0]), bits(got[1][0])) and np.array_equal(bits(got[0][1]), bits(got[1][1]))
    assert got[0][2:] == got[1][2:]


def test_a_wait_that_runs_out_is_done_again_per_step(oracle):
    """No patience at all: the first look that comes too early gives the run
    up, every block leaves, and the per-step kernels give the same result; the
    next run with patience works on the same buffers."""
    case = acquisition(333, 201, 20)
    s, g, vt, vi, wlt = setup_case(oracle, case)
    s.bind_velocity(vt)
    vsrc = np.random.default_rng(5).standard_normal((case.nt, case.ng)).astype(np.float32)
    want_d, want_g = g.forward_modeling(vt, wlt, shot=0), g.calgradient(vt, wlt, vsrc, shot=0)
    for wait_us in (0.0, 5e5, 0.0):
        print(f"wait limit {wait_us} us", flush=True)
        s.set_resident(1, wait_us)
        assert np.array_equal(bits(s.forward_modeling(wlt, shot=0)), bits(want_d))
        assert np.array_equal(bits(s.calgradient(wlt, vsrc, shot=0)), bits(want_g))
