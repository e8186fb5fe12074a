"""time_pass of a batch of tiny FP64 instances times the launches its solves run:
whole iterations, so S advances by 4 * reps of them, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(8, 10, 3), (64, 32, 2), (4, 16, 64)])
def test_times_whole_iterations(hip, shape):
    x, y, z = shape
    X = np.random.default_rng(1).poisson(3.0, (x, y)) + 1.0
    inst = hip.Instance(X=X, z=z, params=hip.Params(1.0, 1.0, [1.0] * x, [1.0] * z), seed=4)
    with hip.Batch([inst], dtype=np.float64, use_psi_appr=False) as b:
        b.solve(3 + 4 * 5)
        ref = b.S(0)
        b.solve(3)
        p, i = b.time_pass(5)
        assert np.array_equal(b.S(0), ref)
        assert 0.0 < p and 0.0 < i
        b.solve(23)
        assert np.array_equal(b.S(0), ref)
