"""The strip-walking forward step of large batches against the CPU oracle:
bit-identical in exact mode, sources, receivers and the boundary band included."""
import numpy as np
import pytest

from swfwi_amd import capi, workloads

from test_gpu_parity import bits, setup_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if capi.device_count() < 1:
        pytest.skip("no HIP device")


# enough entries for the walk (30000 strips x rows), on update regions of one
# strip (nz + nb <= 116), of two with an odd last one, and three; rows (nx + 2 nb)
# that end inside a chunk of 14 or 22; receivers at two depths, coincident
# sources; dt = 2 ms, so that the gradient images from step 151 on
@pytest.mark.parametrize("nx,nz,nb,ns", [(17, 104, 12, 740), (91, 105, 12, 140), (204, 221, 13, 70),
                                         (301, 201, 20, 60)])
def test_batches_bitexact(oracle, nx, nz, nb, ns):
    nt = 170
    sx = (np.arange(ns) * 7 % nx).astype(np.int32)
    sz = (1 + np.arange(ns) % (nz - 1)).astype(np.int32)
    gx = np.concatenate([np.arange(0, nx, 2), [nx - 1, nx - 1]]).astype(np.int32)
    gz = np.concatenate([np.arange(gx.size - 2) % 2 * (nz - 1), [3, 3]]).astype(np.int32)
    case = workloads.Case("strips", nz, nx, 20.0, nb, 0.002, nt, 12.0, sx, sz, gx, gz, 1500.0, 3500.0, seed=nx)
    s, g, vt, vi, wlt = setup_case(oracle, case)
    strips = -(-(nz + nb) // 116)
    assert ns * strips * (nx + 2 * nb) >= 30000
    s.bind_velocity(vt)
    print(f"strip walk {nx}x{nz} nb={nb} shots={ns}", flush=True)
    dobs = s.forward_shots(wlt)
    for shot in (0, ns // 2, ns - 1):
        assert np.array_equal(bits(dobs[shot]), bits(g.forward_modeling(vt, wlt, shot=shot))), shot
    # the band it saves drives the backward run of an epoch: the same gradient
    # as from the per-step kernels of a fixed tile width
    got = []
    for width in (0, 16):
        s.set_tile_x(width)
        s.bind_velocity(vi)
        inv = capi.Inversion(s, wlt, dobs, 1400.0, 3600.0, 3, 200.0)
        inv.fwi_epoch(0)
        got.append((inv.gradient(), s.velocity(), inv.stats()["obj1"], inv.stats()["obj3"]))
        inv.close()
    assert np.count_nonzero(got[0][0]) > 0
    assert np.array_equal(bits(got[0][0]), bits(got[1][0])) and np.array_equal(bits(got[0][1]), bits(got[1][1]))
    assert got[0][2:] == got[1][2:]
