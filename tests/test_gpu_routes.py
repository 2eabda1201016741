"""Which kernels a call runs on (swfwi_solver_last_run), at sizes of every
route, with the seismograms and gradients those kernels give: against the CPU
oracle or against one tiled launch per step, bit for bit."""
import numpy as np
import pytest

from swfwi_amd import capi, workloads

from test_gpu_parity import bits, setup_case
from test_gpu_resident import acquisition

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if capi.device_count() < 1:
        pytest.skip("no HIP device")


def survey(nx, nz, nb, ns, nt=170, precision=capi.PREC_EXACT, gx=None, gz=None, sx=None, sz=None):
    """A solver of ns shots spread over the surface with its true model bound;
    dt = 2 ms, so that the imaging condition starts at step 151."""
    sx = np.linspace(0, nx - 1, ns).astype(np.int32) if sx is None else sx
    sz = (1 + np.arange(ns) % (nz - 1)).astype(np.int32) if sz is None else sz
    gx = np.concatenate([np.arange(0, nx, 3), [nx - 1, nx - 1]]).astype(np.int32) if gx is None else gx
    gz = (np.arange(gx.size) % 2 * (nz - 1)).astype(np.int32) if gz is None else gz
    case = workloads.Case("routes", nz, nx, 20.0, nb, 0.002, nt, 12.0, sx, sz, gx, gz, 1500.0, 3500.0, seed=nx + ns)
    s = capi.Solver(nx, nz, nb, case.dt, case.dx, case.fm, nt, sx, sz, gx, gz, precision)
    v = workloads.models(case)[0]
    s.bind_velocity(capi.expand_domain(v, nb, case.dx, case.dt))
    start = capi.expand_domain(workloads.smoothed(v, 4.0), nb, case.dx, case.dt)
    return case, s, capi.ricker(nt, case.fm, case.dt, 1.0), start


def epoch(s, start, wlt, dobs):
    s.bind_velocity(start)
    inv = capi.Inversion(s, wlt, dobs, 1400.0, 3600.0, 3, 200.0)
    inv.fwi_epoch(0)
    out = inv.gradient(), s.velocity()
    inv.close()
    return out


@pytest.mark.parametrize("nx,nz,nb,nt", [(4, 56, 6, 180), (20, 119, 6, 181), (333, 201, 20, 180), (921, 301, 30, 160),
                                         (1501, 501, 30, 158)])
def test_one_shot_runs_resident(oracle, nx, nz, nb, nt):
    """By rule and without: the loop of one shot is one launch, and a wait that
    runs out is counted."""
    case = acquisition(nx, nz, nb, nt)
    s, g, vt, vi, wlt = setup_case(oracle, case)
    s.bind_velocity(vt)
    assert s.last_run(0)[0] == "none" and s.last_run(1)[0] == "none"
    vsrc = np.random.default_rng(nt).standard_normal((case.nt, case.ng)).astype(np.float32)
    want_d, want_g = g.forward_modeling(vt, wlt, shot=1), g.calgradient(vt, wlt, vsrc, shot=1)
    for mode, route in ((-1, "resident"), (0, "per step"), (1, "resident")):
        print(f"one shot {nx}x{nz} resident {mode}", flush=True)
        s.set_resident(mode)
        assert np.array_equal(bits(s.forward_modeling(wlt, shot=1)), bits(want_d))
        assert s.last_run(0)[:2] == (route, 1 if route == "resident" else nt)
        assert np.array_equal(bits(s.calgradient(wlt, vsrc, shot=1)), bits(want_g))
        assert s.last_run(1)[0] == route and s.last_run(1)[3] == 0
    if nx > 300:  # enough tiles that some block looks too early
        s.set_resident(1, 0.0)
        assert np.array_equal(bits(s.calgradient(wlt, vsrc, shot=1)), bits(want_g))
        assert s.last_run(0)[0] == s.last_run(1)[0] == "per step" and s.last_run(1)[3] == 2
    s.close()


@pytest.mark.parametrize("precision", [capi.PREC_EXACT, capi.PREC_FP32])
@pytest.mark.parametrize("ns,nx,nz,fwd,bwd", [(2, 301, 201, 1, 1), (8, 301, 201, 1, 1), (22, 301, 201, 2, 0),
                                              (13, 301, 201, 1, 2), (79, 120, 90, 2, 0), (60, 120, 90, 1, 0)])
def test_batches_run_resident(ns, nx, nz, fwd, bwd, precision):
    """One launch, or a few where the chip does not hold the batch (bwd 0: two
    at least); the same bits as a tiled launch a step."""
    case, s, wlt, start = survey(nx, nz, 20, ns, precision=precision)
    out = []
    for mode in (0, -1):
        print(f"batch of {ns} on {nx}x{nz}, resident {mode}", flush=True)
        s.set_resident(mode)
        d = s.forward_shots(wlt)
        route = s.last_run(0)
        grad, vel = epoch(s, start, wlt, d)
        back = s.last_run(1)
        s.bind_velocity(capi.expand_domain(workloads.models(case)[0], 20, case.dx, case.dt))
        out.append((d, grad, vel))
        if mode == 0:
            assert route[0] in ("per step", "side by side") and back[0] == "per step"
        else:
            assert route[:2] == ("resident", fwd) and back[0] == "resident" and back[3] == 0
            assert back[1] == bwd if bwd else back[1] >= 2
    for a, b in zip(*out):
        assert np.count_nonzero(a) > 0 and np.array_equal(bits(a), bits(b))
    s.close()


# update regions of exactly one strip (116), of one less full (104), two with an
# odd last one (221) and three (337); chunks of 14 rows, and of 22 from 60000
# strip rows on (more than the ring of 16 holds), the last one partial
@pytest.mark.parametrize("nx,nz,nb,ns,rows", [(205, 104, 12, 140, 14), (205, 92, 12, 300, 22), (301, 201, 20, 60, 14),
                                              (301, 201, 20, 92, 22), (140, 325, 12, 64, 14)])
def test_strip_walks(oracle, nx, nz, nb, ns, rows):
    nt = 170
    case, s, wlt, start = survey(nx, nz, nb, ns, nt)
    g = oracle.Geom(nx, nz, nb, case.dt, case.dx, case.fm, nt, case.sx, case.sz, case.gx, case.gz)
    vt = capi.expand_domain(workloads.models(case)[0], nb, case.dx, case.dt)
    s.set_resident(0)
    print(f"strip walk {nx}x{nz} nb={nb} shots={ns}", flush=True)
    dobs = s.forward_shots(wlt)
    assert s.last_run(0)[:3] == ("strips", nt, rows)
    for shot in (0, ns // 2, ns - 1):
        assert np.array_equal(bits(dobs[shot]), bits(g.forward_modeling(vt, wlt, shot=shot))), shot
    # the band it saves drives the backward run
    got = []
    for width in (0, 16):
        s.set_tile_x(width)
        got.append(epoch(s, start, wlt, dobs))
        assert s.last_run(0)[0] == ("strips" if width == 0 else "per step")
    assert np.count_nonzero(got[0][0]) > 0
    assert all(np.array_equal(bits(a), bits(b)) for a, b in zip(*got))
    s.close()


@pytest.mark.parametrize("precision", [capi.PREC_EXACT, capi.PREC_FP32])
@pytest.mark.parametrize("nx,nz,nb,ns,rows", [(360, 24, 20, 160, 0), (360, 96, 20, 160, 22), (360, 108, 20, 80, 0),
                                              (360, 172, 20, 80, 0), (360, 213, 20, 54, 0), (360, 380, 20, 80, 0),
                                              (360, 511, 20, 16, 0), (360, 511, 20, 31, 22)])
def test_strips_only_where_they_are_filled(nx, nz, nb, ns, rows, precision):
    """Strips hold up to 116 z and tiles 64: the walk takes 2 tiles a strip from
    30000 strip rows, 1.8 from 60000, and never less (one strip of 44, two of 64,
    of 96 and of 100, three of 78, four of 100: tiled)."""
    case, s, wlt, start = survey(nx, nz, nb, ns, nt=12, precision=precision)
    s.set_resident(0)
    strips = -(-(nz + nb) // 116) * (nx + 2 * nb) * ns
    assert strips >= 30000
    print(f"{ns} shots of {nx}x{nz}: {strips} strip rows", flush=True)
    a = s.forward_shots(wlt)
    route = s.last_run(0)
    assert route[:3] == ("strips", 12, rows) if rows else route[:2] == ("per step", 12)
    s.set_tile_x(16)
    assert np.count_nonzero(a) > 0 and np.array_equal(bits(a), bits(s.forward_shots(wlt)))
    s.close()


@pytest.mark.parametrize("members,route", [(60, "strips"), (102, "strips"), (104, "per step")])
def test_strips_of_entries_with_their_own_models(members, route):
    """Members of 201x301: 682 strip rows each, tiled past 70000."""
    from swfwi_amd.enkf import Enkf
    case, s, wlt, start = survey(301, 201, 20, 4, nt=80)
    s.set_resident(0)
    e = Enkf(s, wlt, s.forward_shots(wlt), 0.2, members)
    e.set_members(np.stack([start * np.float32(1 + 0.002 * k) for k in range(members)]))
    print(f"{members} members", flush=True)
    e.analyze(None, 3)
    assert s.last_run(0)[0] == route
    e.close()
    s.close()


@pytest.mark.parametrize("ns,rows", [(60, 14), (92, 22)])
def test_strip_walks_in_fp32(ns, rows):
    case, s, wlt, start = survey(301, 201, 20, ns, precision=capi.PREC_FP32)
    s.set_resident(0)
    print(f"FP32 strip walk, {ns} shots", flush=True)
    a = s.forward_shots(wlt)
    assert s.last_run(0)[:3] == ("strips", case.nt, rows)
    ea = epoch(s, start, wlt, a)
    s.bind_velocity(capi.expand_domain(workloads.models(case)[0], 20, case.dx, case.dt))
    s.set_tile_x(16)
    b = s.forward_shots(wlt)
    assert s.last_run(0)[:3] == ("per step", case.nt, 16)
    eb = epoch(s, start, wlt, b)
    assert np.count_nonzero(a) > 0 and np.array_equal(bits(a), bits(b))
    assert all(np.array_equal(bits(x), bits(y)) for x, y in zip(ea, eb))
    s.close()


@pytest.mark.parametrize("ns,nx,nz,route", [(60, 301, 201, "strips"), (12, 60, 40, "per step")])
def test_captured_loops_replay(ns, nx, nz, route):
    """Graph mode 2 with the resident loop off: the loop is captured and played
    again on the same buffers, with eager work in between, and gives the
    directly launched bits every time."""
    case, s, wlt, start = survey(nx, nz, 20, ns)
    s.set_resident(0)
    s.set_graphs(0)
    direct = s.forward_shots(wlt)
    ge = epoch(s, start, wlt, direct)
    s.set_graphs(2)
    vt = capi.expand_domain(workloads.models(case)[0], 20, case.dx, case.dt)
    for call in range(3):
        print(f"{route} loop in a graph, call {call}", flush=True)
        s.bind_velocity(vt)
        assert np.array_equal(bits(s.forward_shots(wlt)), bits(direct))
        assert s.last_run(0)[0] == route
        s.set_graphs(0)
        s.forward_modeling(wlt, shot=0)  # eager, on the same workspace
        s.set_graphs(2)
        assert all(np.array_equal(bits(a), bits(b)) for a, b in zip(ge, epoch(s, start, wlt, direct)))
    s.close()


def test_crowded_points():
    """More points than a resident tile (512) or a strip walk's unit (64) takes:
    the tiled kernels run, with the same bits."""
    n = 700
    gx = (20 + np.arange(n) % 7).astype(np.int32)
    gz = (np.arange(n) // 7 % 50).astype(np.int32)
    case, s, wlt, start = survey(91, 80, 12, 3, gx=gx, gz=gz)
    vsrc = np.random.default_rng(1).standard_normal((case.nt, n)).astype(np.float32)
    got = []
    for mode in (0, 1):
        s.set_resident(mode)
        print(f"700 receivers in a tile, resident {mode}", flush=True)
        got.append((s.forward_modeling(wlt, shot=1), s.calgradient(wlt, vsrc, shot=1)))
        assert s.last_run(0)[0] == s.last_run(1)[0] == "per step"
    assert all(np.count_nonzero(a) > 0 and np.array_equal(bits(a), bits(b)) for a, b in zip(*got))
    s.close()
    ns = 900
    case, s, wlt, start = survey(17, 104, 12, ns, nt=60, sx=np.full(ns, 8, np.int32),
                                 sz=(np.arange(ns) % 100).astype(np.int32))
    s.set_resident(0)
    print("900 sources in a unit", flush=True)
    a = s.forward_shots(wlt)
    assert s.last_run(0)[0] == "per step"
    s.set_tile_x(16)
    assert np.count_nonzero(a) > 0 and np.array_equal(bits(a), bits(s.forward_shots(wlt)))
    s.close()


def test_tuned_widths_of_the_per_step_loop(oracle):
    """The tuner's widths with the resident loop off, and the rule's without it."""
    case = workloads.small_case(nx=60, nz=40, nb=8, nt=400, ns=3)
    s, g, vt, vi, wlt = setup_case(oracle, case)
    s.bind_velocity(vt)
    s.set_resident(0)
    want = np.stack([g.forward_modeling(vt, wlt, shot=k) for k in range(case.ns)])
    for tuning in (True, False):
        s.set_tuning(tuning)
        print(f"per-step loop, tuning={tuning}", flush=True)
        assert np.array_equal(bits(s.forward_shots(wlt)), bits(want))
        assert s.last_run(0)[0] == "side by side"
        assert all(s.tile_x(k, case.ns) in (8, 16, 32) for k in (0, 1))
        if not tuning:
            assert (s.tile_x(0, case.ns), s.tile_x(1, case.ns)) == (8, 8)
    s.close()


def test_timed_loops_on_lane_streams(oracle):
    """Trial runs side by side on streams (the resident loop off): 20 timed
    epochs pass the pending list's flush size while a lane may still run."""
    case = workloads.small_case(nx=60, nz=40, nb=8, nt=400, ns=3)
    s, g, vt, vi, wlt = setup_case(oracle, case)
    s.bind_velocity(vt)
    s.set_resident(0)
    dobs = s.forward_shots(wlt)
    s.bind_velocity(vi)
    inv = capi.Inversion(s, wlt, dobs, 1400.0, 3600.0, 3, 200.0)
    inv.ess_epoch(0)
    s.set_timing(True)
    n0 = s.counters()[1]
    for it in range(1, 21):
        inv.ess_epoch(it)
        assert s.last_run(0)[0] in ("side by side", "per step") and s.last_run(1)[0] == "per step"
    kt, n1 = s.kernel_times(), s.counters()[1]
    assert kt["fwd"][0] > 0 and kt["bwd"][0] > 0
    assert kt["fwd"][1] == n1[0] - n0[0] and kt["bwd"][1] == n1[1] - n0[1]
    inv.close()
    s.close()
