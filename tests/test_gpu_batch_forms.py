"""The two forms of the batch's step kernel, strips of z walked along x and tiles:
the same bits in every checkpoint format, order and width, and which of them a
batch takes."""
import numpy as np
import pytest

from swfwi_amd import capi
from swfwi_amd.batch import Batch, Group

from test_gpu_batch import models_for

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if capi.device_count() < 1:
        pytest.skip("no HIP device")


def group(nx, nz, nb, ns, nt, **kw):
    sx = np.linspace(0, nx - 1, ns + 2)[1:-1].astype(np.int32)
    return Group(nx=nx, nz=nz, nb=nb, dx=20.0, dt=0.002, fm=12.0, nt=nt, sx=sx, sz=np.ones_like(sx), ng=nx, **kw)


def same(a, b):
    return np.array_equal(np.ascontiguousarray(a).view(np.uint32), np.ascontiguousarray(b).view(np.uint32))


# update regions of one tile and one strip (44, 64), of two (117, 128: two strips
# of 59 and 64), one strip and two tiles (65, 116), five tiles (257); ragged in x
@pytest.mark.parametrize("order", [capi.ORDER_10, capi.ORDER_4])
@pytest.mark.parametrize("snap", [capi.SNAP_F32, capi.SNAP_BF16, capi.SNAP_F16])
@pytest.mark.parametrize("nx,nz,nb", [(33, 37, 7), (61, 57, 7), (70, 58, 7), (40, 109, 7), (131, 110, 7), (20, 121, 7),
                                      (90, 250, 7)])
def test_same_bits(nx, nz, nb, snap, order):
    g = group(nx, nz, nb, 3, 180, nmodels=2)
    b = Batch([g, group(nx + 9, nz + 3, nb, 2, 196)], snap_prec=snap, order=order)
    for gi, gg in enumerate(b.groups):
        for m in range(gg.nmodels):
            b.bind_model(gi, m, models_for(gg, 3 + m)[1])
    dobs = np.random.default_rng(1).standard_normal(b._data_len()).astype(np.float32)
    out = []
    for mode, width in ((0, 16), (0, 24), (0, 32), (1, 16), (1, 32)):
        b.set_strips(mode)
        b.set_tile_x(width)
        print(f"{nx}x{nz} order {order} checkpoints {snap}: strips {mode} width {width}", flush=True)
        d = b.forward()
        b.adjoint_source(dobs, want=False)
        out.append((d, *b.backward(None)))
        assert b.strips() == (mode == 1) and b.tile_x() == width
    assert all(np.count_nonzero(a) > 0 for a in out[0])
    for o in out[1:]:
        assert all(same(x, y) for x, y in zip(out[0], o))
    b.close()


def test_steps_and_taps_in_tiles():
    """step_from and the field taps run in either form."""
    g = group(60, 48, 8, 2, 160)
    b = Batch([g], snap_prec=capi.SNAP_NONE)
    b.bind_model(0, 0, models_for(g, 3)[0])
    prev, cur = np.random.default_rng(2).standard_normal((2, 2) + g.shape).astype(np.float32)
    b.set_taps([4, 20, 39], 1)
    out = []
    for mode in (0, 1):
        b.set_strips(mode)
        print(f"taps, strips {mode}", flush=True)
        b.forward(want_data=False)
        out.append((*b.step_from(prev, cur, 30, 5), *b.taps()))
    assert all(np.count_nonzero(x) > 0 and same(x, y) for x, y in zip(*out))
    b.close()


# one strip, two of 59 and 58 rows, three; odd and even sizes, both row offsets
@pytest.mark.parametrize("order", [capi.ORDER_10, capi.ORDER_4])
@pytest.mark.parametrize("nx,nz,oz", [(33, 37, 0), (34, 38, 1), (41, 109, 0), (40, 109, 1), (70, 244, 1)])
def test_taps_hold_the_field_of_their_step(nx, nz, oz, order):
    """A tap is the field at its step (taken by step_from from the first row of
    data, where the receivers see the source's first sample) at the even points."""
    nb, h, steps = 8, 6, [0, 1, 39, 40]
    g = group(nx, nz, nb, 2, 160, gz=1)
    b = Batch([g], snap_prec=capi.SNAP_NONE, order=order)
    b.bind_model(0, 0, models_for(g, 3)[0])
    b.set_taps(steps, oz)
    for mode in (0, 1):
        b.set_strips(mode)
        print(f"taps {nx}x{nz} order {order} offset {oz}, strips {mode}", flush=True)
        d = b.forward().reshape(g.ns, g.nt, nx)
        taps = b.taps()
        prev, cur = np.zeros((2, g.ns) + g.shape, np.float32)
        for e in range(g.ns):
            cur[e, h + nb + g.sx[e], h + 1] = d[e, 0, g.sx[e]]
        assert np.all(np.count_nonzero(cur, axis=(1, 2)) == 1)
        at = 0
        for k, step in enumerate(steps):
            if step > at:
                prev, cur = (f.reshape((g.ns,) + g.shape) for f in b.step_from(prev, cur, at, step - at))
                at = step
            for e in range(g.ns):
                want = np.zeros_like(taps[e][k])
                inner = cur[e, h:-h, h + oz:-h][::2, ::2][:want.shape[0] - h, :want.shape[1] - h]
                want[h:, h:][:inner.shape[0], :inner.shape[1]] = inner
                assert same(taps[e][k], want), (mode, step, e)
    b.close()


@pytest.mark.parametrize("nx,nz,nb,ns,order,strips", [
    (270, 49, 15, 12, capi.ORDER_10, True),    # 64 z, 3600 strip rows: too few waves for tiles to pay
    (270, 49, 15, 48, capi.ORDER_10, False),   # 14400: 0.83 of the tiles' speed as strips
    (270, 113, 15, 48, capi.ORDER_10, False),  # 128 z: two half-empty strips
    (270, 109, 15, 48, capi.ORDER_4, True),    # 124 z fill a strip of the 4th-order step
    (270, 113, 15, 48, capi.ORDER_4, False),
    (270, 75, 15, 48, capi.ORDER_10, True),    # 90 z: two tiles a strip
    (670, 49, 15, 96, capi.ORDER_10, True),    # 64 z, 67200 strip rows: 1.1
    (270, 125, 15, 48, capi.ORDER_10, True),   # 140 z: three tiles in two strips
])
def test_the_form_a_batch_takes(nx, nz, nb, ns, order, strips):
    b = Batch([group(nx, nz, nb, ns, 160)], snap_prec=capi.SNAP_NONE, order=order)
    assert b.strips() == strips
    b.set_strips(0 if strips else 1)
    assert b.strips() != strips
    b.set_strips(-1)
    assert b.strips() == strips
    b.close()
