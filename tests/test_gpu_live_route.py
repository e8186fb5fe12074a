"""Batches over packed nonempty fibers against the dense passes, bit for bit, with
the route asserted: the packed batch takes more device memory than the dense one
of the same problem. A smallest denormal in one empty fiber's S0 keeps that batch
dense without changing a sum (tests/test_gpu_live.py). Beside solve: solve_tol,
which scores in between and goes on, fact from the partial sums, and time_pass,
which runs passes without their prep. FP64 tiles as tall as the table allows have
more fibers than fit the LDS whole, so their partial sums run over k in parts."""
import numpy as np
import pytest

from test_gpu_live import SHAPES, _problem

pytestmark = pytest.mark.gpu

PARTS = [(256, 130, 31), (200, 129, 32), (131, 70, 45), (150, 200, 64)]


def _pair(hip, shape, share, dt, algo=0, appr=True, more=()):
    x, y, z = shape
    X, alpha, beta, S0, dense = _problem(x, y, z, share, dt, x + z)
    p = hip.Params(1.0, 1.0, alpha, beta)
    a, b = ([hip.Instance(X=X, z=z, params=p, S0=s)] + list(more) for s in (S0, dense))
    kw = dict(dtype=dt, use_psi_appr=appr, algo=algo)
    a, b = hip.Batch(a, **kw), hip.Batch(b, **kw)
    assert a.info()["device_bytes"] > b.info()["device_bytes"], (shape, share, "not packed")
    return a, b


def _equal(a, b, what):
    for u, v in zip(a, b):
        u, v = np.asarray(u), np.asarray(v)
        assert np.all(np.isfinite(u)) and np.array_equal(u, v), what


def _check(hip, shape, dt, shares, more=()):
    for share in shares:
        for algo, appr in [(hip.ALGO_MULT, True), (hip.ALGO_ADD, True)] + [(hip.ALGO_MULT, False)] * (dt == np.float64):
            a, b = _pair(hip, shape, share, dt, algo, appr, more)
            what = (shape, share, algo, appr)
            with a, b:
                a.solve(7), b.solve(7)
                _equal([a.S(0)], [b.S(0)], what)
                assert a.S(0).any()
                _equal(a.fact(0), b.fact(0), what + ("fact",))
                # (a solve that no longer changes ends at a tolerance of 0)
                assert a.solve_tol(8, 0.0, 3)[0] == b.solve_tol(8, 0.0, 3)[0]
                _equal([a.S(0), a.log_marginal()], [b.S(0), b.log_marginal()], what + ("solve_tol",))
                # passes on stale gradients: S may end as NaN, in both
                a.time_pass(2), b.time_pass(2)
                assert np.array_equal(a.S(0), b.S(0), equal_nan=True), what + ("time_pass",)
                a.solve(7), b.solve(7)
                _equal([a.S(0)], [b.S(0)], what + ("again",))


@pytest.fixture(scope="module")
def large(hip):
    """Takes a batch past the total at which FP32 instances of z <= 4 are packed."""
    X = (np.random.default_rng(0).random((800, 800)) < 0.02).astype(np.float32)
    return hip.Instance(X=X, z=12, params=hip.Params(1.0, 1.0, [1.0] * 800, [1.0] * 12), seed=1)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_packed_batch_equals_dense(hip, large, shape, dt):
    _check(hip, shape, dt, (0.03, 0.2, 0.3), [large] if dt == np.float32 and shape[2] <= 4 else ())


@pytest.mark.parametrize("shape", PARTS)
def test_sums_in_parts_fp64(hip, shape):
    x, y, z = shape
    old = hip.tune_get(np.float64, z, x * y)
    try:
        hip.tune_set(np.float64, z, x * y, 64)
        _check(hip, shape, np.float64, (0.03, 0.3))
    finally:
        hip.tune_set(np.float64, z, x * y, old)
