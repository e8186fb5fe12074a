"""Step passes over the packed nonempty fibers against the dense passes.

An instance whose S0 holds anything in a fiber with X = 0 is not packed. The
smallest denormal there changes no sum (every S_i+k and S_+jk gets alpha or
beta >= 1 added) and the first step clears it, so the same problem runs both
ways; the packed step does the dense one's operations in its order, so the
results are equal bit for bit. Shapes: ragged tiles, z of every residue mod 4
and of every FP64 lane split, tiles with no fiber, with enough fibers that the
partial sums run over k in parts, and X with whole rows and columns empty."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(37, 70, 1), (65, 33, 2), (70, 131, 3), (100, 100, 4), (129, 65, 7), (90, 90, 8), (33, 200, 12),
          (100, 100, 17), (140, 100, 18), (77, 190, 24), (256, 130, 31), (200, 129, 32), (60, 65, 33),
          (131, 70, 45), (130, 140, 63), (150, 200, 64)]


def _problem(x, y, z, share, dt, seed):
    rng = np.random.default_rng(seed)
    X = (rng.poisson(3.0, (x, y)) + 1.0) * (rng.random((x, y)) < share)
    X[rng.integers(x)] = 0.0
    X[:, rng.integers(y)] = 0.0
    X[0, 0], X[-1, -1] = 0.0, 12.0  # S + 1 >= 10: the FP64 digamma's other branch
    S0 = X[:, :, None] * rng.dirichlet(np.full(z, 0.3), size=(x, y))
    alpha, beta = rng.uniform(0.5, 2.0, x), rng.uniform(1.0, 2.0, z)
    dense = S0.astype(dt)
    dense[0, 0, 0] = np.nextafter(dt(0), dt(1))
    return X.astype(dt), alpha, beta, S0.astype(dt), dense


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_packed_equals_dense(hip, shape, dt):
    x, y, z = shape
    for share in (0.03, 0.2, 0.45):
        X, alpha, beta, S0, dense = _problem(x, y, z, share, dt, x + z)
        p = hip.Params(1.0, 1.0, alpha, beta)
        for appr in ([True] if dt == np.float32 else [False, True]):
            a = hip.bld_mult(X, z, p, 7, appr, S0=S0, dtype=dt)
            b = hip.bld_mult(X, z, p, 7, appr, S0=dense, dtype=dt)
            assert np.all(np.isfinite(a)) and a.any()
            assert np.array_equal(a, b), ("mult", share, appr, np.abs(a - b).max())
        a = hip.bld_add(X, z, p, 5, S0=S0, dtype=dt)
        b = hip.bld_add(X, z, p, 5, S0=dense, dtype=dt)
        assert np.all(np.isfinite(a)) and a.any()
        assert np.array_equal(a, b), ("add", share, np.abs(a - b).max())
