"""A served request of no iterations gives back its S0, whatever earlier requests
left in the server's memory: here NaN everywhere, from a request that did the
same with an S0 of NaN."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("given", [True, False])
def test_zero_iterations_on_used_memory(hip, dtype, given):
    x, y, z = 96, 80, 12
    rng = np.random.default_rng(2)
    X = ((rng.poisson(3.0, (x, y)) + 1.0) * (rng.random((x, y)) < 0.1)).astype(dtype)
    p = hip.Params(20.0, 1.0, [1.0] * x, [1.0] * z)
    S0 = (X[:, :, None] * rng.dirichlet(np.ones(z), size=(x, y))).astype(dtype)
    inst = hip.Instance(X=X, z=z, params=p, S0=S0 if given else None, seed=7)
    big = (4 * x, 4 * y, z)
    nan = hip.Instance(X=np.ones(big[:2], dtype), z=z, params=hip.Params(20.0, 1.0, [1.0] * big[0], [1.0] * z),
                       S0=np.full(big, np.nan, dtype))
    with hip.Batch([inst], dtype=dtype) as b:
        b.solve(0)
        ref, lm = b.S(0), b.log_marginal()[0]
    with hip.Server(2 * hip.Server.request_bytes(big, dtype), dtype=dtype) as srv:
        t = srv.submit(nan, 0)
        srv.wait(t)
        assert np.all(np.isnan(srv.collect(t)[0]))
        t = srv.submit(inst, 0, log_marginal=True)
        srv.wait(t)
        S, got, _ = srv.collect(t)
    assert np.array_equal(S, ref)
    assert got == pytest.approx(lm, rel=1e-14)
