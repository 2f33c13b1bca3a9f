"""Device orthonormalisation (mq_orthonormalise, the step of the Jacobi-Davidson driver):
basis sizes around the groups of eight vectors and one wave's rows, vectors below and above
one block's threads, and vectors that lose so much of their norm that the second
Gram-Schmidt pass runs and its norm is used."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps / 2
SHAPES = [(1, 0), (2, 1), (63, 7), (300, 8), (513, 9), (1330, 33), (2000, 130), (65536, 16), (70001, 41), (140001, 4)]


def _basis(n, m, seed):
    rng = np.random.default_rng(seed)
    q = np.linalg.qr(rng.standard_normal((n, m + 1)))[0].T.copy()
    return q[:m], q[m], rng


def _bound(m):
    """|V t| and the error of |t| after a pass that kept a quarter of the norm at least: a dot
    product's sums are at most 40 additions deep, an update adds m products."""
    return 4 * (40 + 2 * m) * EPS


@pytest.mark.parametrize("n,m", SHAPES)
def test_one_pass(gpu_engine, n, m):
    print(f"n {n} m {m}", flush=True)
    V, w, rng = _basis(n, m, n + m)
    # half of t lies in V: no second pass
    c = rng.standard_normal(m)
    t = 3.0 * (w + (c / np.linalg.norm(c) @ V if m else 0.0))
    got = gpu_engine.orthonormalise(gpu_engine.to_dev(V), gpu_engine.to_dev(t)).cpu().numpy()
    assert abs(np.linalg.norm(got) - 1) <= _bound(m)
    assert np.abs(V @ got).max(initial=0.0) <= _bound(m)
    assert np.linalg.norm(got - w) <= _bound(m) * np.sqrt(m + 1) + 8 * EPS


@pytest.mark.parametrize("n,m", [s for s in SHAPES if s[1] > 0])
def test_second_pass(gpu_engine, n, m):
    print(f"n {n} m {m}", flush=True)
    V, w, rng = _basis(n, m, 7 * n + m)
    c = rng.standard_normal(m)
    drop = 1e-11
    t = (c / np.linalg.norm(c)) @ V + drop * w
    # one pass leaves rounding errors of t in V, a 1e-5th of what remains: without a second one,
    # or with the first one's norm, the bounds below are missed by orders of magnitude
    one = t - (V @ t) @ V
    assert np.linalg.norm(one) <= 0.25 * np.linalg.norm(t)
    got = gpu_engine.orthonormalise(gpu_engine.to_dev(V), gpu_engine.to_dev(t)).cpu().numpy()
    assert abs(np.linalg.norm(got) - 1) <= _bound(m)
    assert np.abs(V @ got).max() <= _bound(m)
    # the direction is known to the rounding of t's own elements
    assert np.linalg.norm(got - w) <= (4 + 2 * m) * EPS * np.sqrt(2.0) / drop


def test_argument_errors(gpu_engine):
    from qcmaquis_amd.gpu import lib
    t = gpu_engine.to_dev(np.ones(4))
    assert lib().mq_orthonormalise(gpu_engine.ctx, None, 4, 1, t.data_ptr()) != 0
    assert lib().mq_orthonormalise(gpu_engine.ctx, None, 0, 0, t.data_ptr()) != 0
    assert lib().mq_orthonormalise(gpu_engine.ctx, None, 4, 0, None) != 0
    with pytest.raises(ValueError):
        gpu_engine.orthonormalise(gpu_engine.to_dev(np.ones((2, 5))), t)
