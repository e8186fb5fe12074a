"""Instances of depth 0: S has no elements, and every entry point that takes
such an instance plans it as it plans x = 0 or y = 0. Each planner runs in a
process of its own, so that one that ends the process fails its test only."""
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("call", ["hip.Server.request_bytes((10, 7, 0), np.{0})", "hip.Server.request_bytes((2000, 1, 0), np.{0})"])
def test_planner(dtype, call):
    code = "import numpy as np, bnmf_hip as hip; print(" + call.format(dtype) + ")"
    r = subprocess.run([sys.executable, "-c", code], cwd=os.path.join(ROOT, "bnmf-algs_amd"), capture_output=True,
                       text=True, timeout=120)
    assert r.returncode == 0, (r.returncode, r.stderr[-300:])
    assert int(r.stdout) >= 4


class _Inst:
    def __init__(self, hip, x, y, z, dtype):
        self.X = np.random.default_rng(x).poisson(2.0, (x, y)).astype(dtype)
        self.z, self.seed, self.S0 = z, 3, None
        self.params = hip.Params(4.0, 1.0, [1.0] * x, [1.0] * z)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_on_device(hip, dtype):
    empty, full = _Inst(hip, 10, 7, 0, dtype), _Inst(hip, 40, 50, 6, dtype)
    with hip.Batch([full], dtype=dtype) as b:
        b.solve(5)
        ref, lm = b.S(0), b.log_marginal()[0]
    with hip.Batch([empty, full], dtype=dtype) as b:
        b.solve(5)
        assert b.S(0).size == 0 and np.array_equal(b.S(1), ref)
        assert np.array_equal(b.log_marginal(), [0.0, lm])
    with hip.Server(1 << 26, dtype=dtype) as srv:
        tickets = [srv.submit(i, 5) for i in (empty, full)]
        for t, r in zip(tickets, (np.empty((10, 7, 0)), ref)):
            srv.wait(t)
            assert np.array_equal(srv.collect(t)[0], r)
    assert hip.log_marginal_S(np.empty((10, 7, 0), dtype), empty.params) == 0.0
