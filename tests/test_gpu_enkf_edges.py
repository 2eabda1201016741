"""The analysis kernels of the ensemble Kalman filter where their member chunks
and data rows end, against the numpy oracle."""
import numpy as np
import pytest

from oracle import enkf_oracle as eo
from swfwi_amd import capi, workloads
from swfwi_amd.enkf import Enkf

from test_enkf import _ensemble

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,nt", [(2, 341), (16, 340), (17, 400), (113, 340)])
def test_gpu_enkf_analysis_at_chunk_edges(oracle, N, nt):
    """Ensembles of one member chunk of the update, one more, and past the
    112 of the matrix-core products; data rows that leave remainders.  The
    tolerances of the analysis above."""
    if capi.device_count() < 1:
        pytest.skip("no HIP device")
    case = workloads.small_case(nx=21, nz=17, nb=6, nt=nt, ns=2)
    vtrue, members = _ensemble(case, N, 5)
    wlt = capi.ricker(case.nt, case.fm, case.dt, 1.0)
    s = capi.Solver(case.nx, case.nz, case.nb, case.dt, case.dx, case.fm, case.nt, case.sx, case.sz, case.gx,
                    case.gz)
    s.bind_velocity(capi.expand_domain(vtrue, case.nb, case.dx, case.dt))
    dobs = s.forward_shots(wlt)
    e = Enkf(s, wlt, dobs, 0.2, N)
    e.set_members(members)
    rms = float(np.sqrt(np.mean(dobs.astype(np.float64) ** 2)))
    E = np.random.default_rng(6).standard_normal((N, case.nt, case.ng)) * 0.05 * rms
    e.analyze(E)
    code = oracle.gen_codes(2, case.ns)
    g = oracle.Geom(case.nx, case.nz, case.nb, case.dt, case.dx, case.fm, case.nt, case.sx, case.sz, case.gx,
                    case.gz)
    enc = oracle.encode_source(code, wlt)
    ha = np.stack([g.forward_modeling(members[i], enc, shot=-1) for i in range(N)])
    want, mid = eo.analyze(members, ha, oracle.encode_obs(code, dobs), E, case.dx, case.dt, sigfac=0.2)
    info = e.info()
    assert info["clip"] == mid["clip"]
    assert np.abs(info["gain"] - mid["t4"]).max() <= 1e-6 * np.abs(mid["t4"]).max()
    got = e.members()
    rel = np.abs(got.astype(np.float64) - want) / np.abs(want)
    print(f"enkf N={N}: members {rel.max():.2e}", flush=True)
    assert rel.max() < 1e-5
    assert np.abs(got - members).max() > 0
    e.close()
    s.close()
