"""A request that fits beside the dense tensors of an active one starts at once,
though that one's packed fibers are in the way: they are given back in the middle
of its solve, and both results are those of a batch, bit for bit."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _inst(hip, x, y, z, dtype, seed):
    rng = np.random.default_rng(seed)
    X = ((rng.poisson(3.0, (x, y)) + 1.0) * (rng.random((x, y)) < 0.1)).astype(dtype)
    return hip.Instance(X=X, z=z, params=hip.Params(1.0, 1.0, [1.0] * x, [1.0] * z), seed=seed)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_later_request_does_not_wait(hip, dtype):
    a, b = _inst(hip, 300, 250, 24, dtype, 1), _inst(hip, 220, 250, 24, dtype, 2)
    long, short = 40000, 50
    need = [hip.Server.request_bytes((i.X.shape[0], i.X.shape[1], i.z), dtype) for i in (a, b)]
    ref = []
    for i, it in ((a, long), (b, short)):
        with hip.Batch([i], dtype=dtype) as batch:
            batch.solve(it)
            ref.append(batch.S(0))
    with hip.Server(sum(need), dtype=dtype) as srv:
        ta = srv.submit(a, long)
        end = time.time() + 20
        while srv.stats()["bytes_in_use"] <= need[0]:
            assert time.time() < end, "not packed"
        tb = srv.submit(b, short)
        assert srv.wait(tb, 30.0) == hip.OK
        assert not srv.poll(ta)
        assert np.array_equal(srv.collect(tb)[0], ref[1])
        assert srv.wait(ta, 60.0) == hip.OK
        assert np.array_equal(srv.collect(ta)[0], ref[0])
        st = srv.stats()
        assert st["peak_active"] == 2 and st["bytes_in_use"] == 0
