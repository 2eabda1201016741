"""The training step's kernels at the sizes where their tiles end, and its
two launches against the parts they stand for.

* the weight gradient (sums over the tile's points on the matrix cores) for
  regions of one point, of exactly one tile and two tiles with their 2-cell
  margin, and one point more, against the oracle with the same BF16
  roundings.  Tolerance: a value at a rounding tie may go to the other BF16
  neighbour (2^-9 relative in one of the 144 terms of a sum), well below 2e-3
  of the gradient's norm;
* the minibatch read in place: with a step length of 0 the losses over one
  pass are the samples' own losses, in some order;
* Adam's step where the sums end: the first step is -lr g / (|g| + eps), and
  the trained net gives the bits of a new net with its weights, so that
  every packed form was renewed."""
import numpy as np
import pytest

from oracle import convnet as cn
from swfwi_amd import capi
from swfwi_amd.batch import Net

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if capi.device_count() < 1:
        pytest.skip("no HIP device")


def stack(seed, e, nx, nz):
    from scipy.ndimage import gaussian_filter
    r = np.random.default_rng(seed)
    f = lambda: np.stack([gaussian_filter(r.standard_normal((nx, nz)), 2.0) for _ in range(e)])  # noqa: E731
    p = f()
    p = (p / np.abs(p).max()).astype(np.float32)
    q = f()
    rv = r.uniform(0.05, 0.3, p.shape).astype(np.float32)
    return p, rv, (p + 0.05 * q / np.abs(q).max()).astype(np.float32)


@pytest.mark.parametrize("sx,sz,e", [(1, 1, 1), (12, 28, 2), (13, 29, 3), (28, 12, 1), (45, 1, 2)])
def test_gradient_at_tile_edges(sx, sz, e):
    p, rv, t = stack(sx * 100 + sz, e, sx + 10, sz + 11)
    region = (5, 5 + sx, 5, 5 + sz)
    theta = Net.initial(seed=7, scale=0.1)
    net = Net(theta)
    loss, g = net.loss_grad(p, rv, t, region)
    net.close()
    wl, wg = cn.loss_grad(p, rv, t, theta, region, emulate=True)
    assert abs(loss - wl) <= 1e-4 * wl
    n1, n2 = cn.NW1, 9 * 16 * 16
    for name, sl in (("W1", slice(0, n1)), ("W2", slice(n1, n1 + n2)), ("W3", slice(n1 + n2, cn.NPARAMS))):
        err = np.linalg.norm(g[sl] - wg[sl]) / np.linalg.norm(wg[sl])
        print(f"{sx} x {sz} x {e}, d loss / d {name}: rel-L2 {err:.2e}", flush=True)
        assert err < 2e-3, name


def test_minibatches_read_in_place():
    p, rv, t = stack(3, 5, 40, 33)
    region = [6, 33, 5, 27]
    theta = Net.initial(seed=9, scale=0.1)
    net = Net(theta)
    each = [net.loss_grad(p[k:k + 1], rv[k:k + 1], t[k:k + 1], region)[0] for k in range(5)]
    net.set_data(p, rv, t, region)
    one = net.train(1, 5, 0.0, 4)
    np.testing.assert_allclose(np.sort(one), np.sort(each), rtol=1e-12)
    pair = net.train(2, 5, 0.0, 4)  # two passes over the five samples
    np.testing.assert_allclose(pair.sum(), np.sum(each), rtol=1e-12)
    assert np.array_equal(net.weights(), theta)
    net.close()


def test_adam_step_and_packed_weights():
    p, rv, t = stack(5, 4, 40, 33)
    region = [6, 33, 5, 27]
    theta = Net.initial(seed=11, scale=0.1)
    net = Net(theta)
    _, g = net.loss_grad(p, rv, t, region)
    net.set_data(p, rv, t, region)
    lr = 1e-3
    net.train(4, 1, lr, 1)
    now = net.weights()
    # the sums run in another order of the samples: a gradient above 1e-3 of
    # the largest keeps its sign, and eps = 1e-8 bends the step by < 1e-2
    big = np.abs(g) > 1e-3 * np.abs(g).max()
    want = theta.astype(np.float64) - lr * g / (np.abs(g) + 1e-8)
    assert big.sum() > 1000
    assert np.abs(now - want)[big].max() < 2e-2 * lr
    net.train(3, 7, lr, 2)
    y = net.apply(p, rv, region)
    other = Net(net.weights())
    assert np.array_equal(y, other.apply(p, rv, region))
    la, ga = net.loss_grad(p, rv, t, region)
    lb, gb = other.loss_grad(p, rv, t, region)
    assert la == lb and np.array_equal(ga, gb)
    other.close()
    net.close()
