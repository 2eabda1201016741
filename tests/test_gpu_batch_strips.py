"""The batch's step kernel at the edges of its strips (116 or 124 z) and of its
chunks of rows: seismograms against the CPU oracle, gradients and the
4th-order stencil against a float64 leapfrog written from the formulas (the
gradient with the batch's own imaging condition, every 4th step with weight 4).

Tolerances are the FP32 budgets: seismogram and fields 1e-5, gradient 1e-4."""
import numpy as np
import pytest

from swfwi_amd import capi
from swfwi_amd.batch import Batch, Group

from test_gpu_batch import SEIS_TOL, models_for, rel_l2

pytestmark = pytest.mark.gpu

GRAD_TOL = 1e-4
A = [float(np.float32(a)) for a in (1.53400796, 1.78858721, -0.31660756, 0.07612173, -0.01626042, 0.00216736)]


class Leapfrog:
    """The damped step on [entries][nxpad][nzpad] float64 fields."""

    def __init__(self, vel, nb, order):
        w, self.order = nb + 6, order
        d = np.zeros(vel.shape)
        k = np.arange(w)
        d[:w] = (0.05 * ((w - k) / w) ** 2)[:, None]
        d[vel.shape[0] - w:] = (0.05 * ((k + 1) / w) ** 2)[:, None]
        d[:, vel.shape[1] - w:] = (0.05 * ((k + 1) / w) ** 2)[None, :]
        d = d[6:-6, 6:-6]
        self.a, self.b, self.r = 2 - 2 * d + d * d, 1 - 2 * d, 1.0 / vel.astype(np.float64)[6:-6, 6:-6]

    def step(self, c, p):
        """the next field; its 6-cell rim keeps what p holds"""
        at = lambda i, j: c[:, 5 + i:c.shape[1] - 5 + i, 5 + j:c.shape[2] - 5 + j]  # noqa: E731
        w = [-4 * A[0]] + A[1:] if self.order == 10 else [-5.0, 4.0 / 3, -1.0 / 12]
        u = w[0] * at(0, 0)
        for k in range(1, len(w)):
            u = u + w[k] * (at(0, -k) + at(0, k) + at(-k, 0) + at(k, 0))
        n = p.copy()
        i = u[:, 1:-1, 1:-1]
        v = self.a * c[:, 6:-6, 6:-6] - self.b * p[:, 6:-6, 6:-6] + self.r * i
        if self.order == 10:
            v = v + self.r ** 2 / 12 * (u[:, 1:-1, :-2] + u[:, 1:-1, 2:] + u[:, :-2, 1:-1] + u[:, 2:, 1:-1] - 4 * i)
        n[:, 6:-6, 6:-6] = v
        return n


def gradients64(g, vel, wlt, vsrc):
    """Per-shot gradients of a group with one model from its adjoint sources."""
    f, bx, n = Leapfrog(vel, g.nb, 10), g.nb + 6, len(g.sx)
    e = np.arange(n)
    weight = lambda it: 4.0 * min(max((g.dt * it - 0.3) / 0.1, 0.0), 1.0)  # noqa: E731
    last = min(it for it in range(4, g.nt, 4) if float(np.float32(g.dt)) * it > 0.3)
    c, p, snap = np.zeros((n,) + g.shape), np.zeros((n,) + g.shape), {}
    c[e, g.sx + bx, g.sz + 6] += wlt[0]
    for it in range(g.nt):
        snap[it] = c
        c, p = f.step(c, p), c
        if it + 1 < g.nt:
            c[e, g.sx + bx, g.sz + 6] += wlt[it + 1]
    c, p, grad = np.zeros((n,) + g.shape), np.zeros((n,) + g.shape), np.zeros((n,) + g.shape)
    rec = (slice(None), slice(bx + g.gx0, bx + g.gx0 + g.ng), g.gz + 6)
    c[rec] += vsrc[:, g.nt - 1]
    inner = (slice(None), slice(6, -6), slice(6, -6))
    for it in range(g.nt - 1, last - 1, -1):
        if it % 4 == 0:
            grad[inner] -= weight(it) * snap[it - 1][inner] * c[inner]
        c, p = f.step(c, p), c
        if it - 1 >= last:
            c[rec] += vsrc[:, it - 1]
    return grad


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if capi.device_count() < 1:
        pytest.skip("no HIP device")


def group(nx, nz, nb, nt=340, **kw):
    sx = np.array([0, nx - 1], np.int32)
    sz = np.array([1, nz - 1], np.int32)
    return Group(nx=nx, nz=nz, nb=nb, dx=10.0, dt=0.001, fm=20.0, nt=nt, sx=sx, sz=sz, **kw)


# update regions nz + nb of one strip (20: narrower than a wave), 116, 117 (two
# strips, an odd last one), 232, 233 (three); nx + 2 nb of less than a chunk up
# to many, not multiples of 6, 10 or 14; receivers in the first strip and beyond
@pytest.mark.parametrize("nx,nz,nb,gz,width", [(5, 14, 6, 0, 16), (20, 110, 6, 3, 24), (21, 111, 6, 110, 32),
                                               (64, 226, 6, 116, 0), (131, 227, 6, 0, 32)])
def test_strip_edges_against_oracles(oracle, nx, nz, nb, gz, width):
    g = group(nx, nz, nb, ng=nx, gz=gz)
    b = Batch([g], snap_prec=capi.SNAP_F32)
    b.set_tile_x(width)
    vt, vi = models_for(g, nz)
    b.bind_model(0, 0, vt)
    dobs = b.forward()
    b.bind_model(0, 0, vi)
    D = b.split_data(b.forward())
    V = b.split_data(b.adjoint_source(dobs))
    GE = b.split_grid(b.backward(None, want_entries=True, want_models=False)[0])
    og = oracle.Geom(nx, nz, nb, g.dt, g.dx, g.fm, g.nt, g.sx, g.sz, np.arange(nx, dtype=np.int32),
                     np.full(nx, gz, np.int32))
    wlt = oracle.ricker(g.nt, g.fm, g.dt, 1.0)
    print(f"strips {nx}x{nz} nb={nb} gz={gz} width {b.tile_x()}", flush=True)
    want = gradients64(g, vi, wlt, np.stack(V).astype(np.float64))
    for s in range(2):
        assert rel_l2(D[s], og.forward_modeling(vi, wlt, shot=s)) <= SEIS_TOL
    # over both shots: where a shot's waves do not reach the receivers in 340
    # steps, its own gradient lies below FP32's smallest values
    assert rel_l2(np.stack(GE), want) <= GRAD_TOL
    b.close()


@pytest.mark.parametrize("nx,nz,nb", [(30, 118, 6), (31, 119, 6), (90, 243, 7)])
def test_fourth_order_steps_against_float64(nx, nz, nb):
    """step_from of the 4th-order stencil: 6 damped steps of two random entries
    (float32 rounding of 6 steps of O(1) values stays below 1e-5)."""
    g = group(nx, nz, nb, nt=320)
    b = Batch([g], snap_prec=capi.SNAP_NONE, order=capi.ORDER_4)
    vt, _ = models_for(g, 3)
    b.bind_model(0, 0, vt)
    rng = np.random.default_rng(nx)
    prev, cur = rng.standard_normal((2, 2) + g.shape).astype(np.float32)
    it0 = 310  # the Ricker amplitudes are over
    print(f"4th order {nx}x{nz} nb={nb}", flush=True)
    po, co = b.step_from(prev, cur, it0, 6)
    p, c = prev.astype(np.float64), cur.astype(np.float64)
    f = Leapfrog(vt, nb, 4)
    for _ in range(6):
        c, p = f.step(c, p), c
    assert rel_l2(co.reshape(c.shape), c) <= SEIS_TOL
    assert rel_l2(po.reshape(p.shape), p) <= SEIS_TOL
    b.close()
