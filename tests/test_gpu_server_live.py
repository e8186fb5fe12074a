"""Served requests over packed nonempty fibers: the same bits whether the arena
has room for their lists, has not, or a batch solves them; iteration counts that
end in different steps, both depths of launch, S0 given and drawn, dense requests
beside them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(150, 90, 7, 0.05), (70, 131, 33, 0.1), (64, 64, 64, 0.02), (40, 300, 17, 0.3), (33, 20, 5, 0.9), (200, 60, 3, 0.0)]


class _Inst:
    def __init__(self, hip, n, dtype):
        x, y, z, share = SHAPES[n]
        rng = np.random.default_rng(n)
        self.X = ((rng.poisson(3.0, (x, y)) + 1.0) * (rng.random((x, y)) < share)).astype(dtype)
        self.S0 = None if n % 2 else (self.X[:, :, None] * rng.dirichlet(np.ones(z), size=(x, y))).astype(dtype)
        self.z, self.seed = z, 40 + n
        self.params = hip.Params(20.0, 1.0, [1.0] * x, [1.0] * z)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_server_packed_equals_batch(hip, dtype):
    insts = [_Inst(hip, n, dtype) for n in range(len(SHAPES))]
    iters = [20, 3, 17, 8, 9, 5]
    ref = []
    for i, it in zip(insts, iters):
        with hip.Batch([i], dtype=dtype) as b:
            b.solve(it)
            ref.append(b.S(0))
    dt = hip.F32 if dtype == np.float32 else hip.F64
    sizes = [hip.lib().bnmf_server_request_bytes(dt, *s[:3]) for s in SHAPES]
    for budget in (max(sizes), 2 * sum(sizes) + (1 << 20)):
        with hip.Server(budget, dtype=dtype) as srv:
            tickets = [srv.submit(i, it) for i, it in zip(insts, iters)]
            for t, r, s in zip(tickets, ref, SHAPES):
                srv.wait(t)
                assert np.array_equal(srv.collect(t)[0], r), (s, budget)
            assert srv.stats()["bytes_in_use"] == 0
