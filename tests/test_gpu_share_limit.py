"""Which instances are packed, by their share of nonempty entries: device memory
shows it. Shares on both sides of where a packed and a dense iteration take the
same time."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# dtype, algo (0 mult, 1 add), x, y, z, instances, a share that pays, one that does not
CASES = [
    (np.float32, 0, 2048, 2048, 64, 1, 0.25, 0.4),
    (np.float32, 0, 1024, 1024, 64, 1, 0.35, 0.49),
    (np.float32, 0, 1024, 1024, 32, 1, 0.4, 0.49),
    (np.float32, 0, 256, 256, 32, 1, 0.3, 0.45),
    (np.float32, 1, 256, 256, 64, 1, 0.3, 0.45),
    (np.float32, 0, 100, 100, 17, 1, 0.45, 0.6),
    (np.float32, 0, 512, 512, 4, 8, 0.3, 0.6),
    (np.float32, 0, 128, 128, 4, 1, None, 0.05),
    (np.float64, 0, 1024, 1024, 32, 1, 0.25, 0.4),
    (np.float64, 0, 2048, 2048, 32, 1, 0.2, 0.35),
    (np.float64, 0, 256, 256, 32, 1, 0.3, 0.45),
    (np.float64, 1, 256, 256, 32, 1, 0.45, 0.6),
]


@pytest.mark.parametrize("case", CASES)
def test_limit(hip, case):
    dt, algo, x, y, z, n, pays, loses = case
    rng = np.random.default_rng(1)
    U = rng.random((x, y))
    p = hip.Params(1.0, 1.0, [1.0] * x, [1.0] * z)

    def memory(share, eps):
        X = (U < share).astype(dt)
        with hip.Batch([hip.Instance(X=X, z=z, params=p, seed=k) for k in range(n)], dtype=dt, algo=algo, eps=eps) as b:
            return b.info()["device_bytes"]
    # eps below 1e-200 is not for the packed form
    assert memory(loses, 1e-50) == memory(loses, 1e-250)
    assert pays is None or memory(pays, 1e-50) > memory(pays, 1e-250)


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_in_company(hip, dt):
    """An instance past its own limit is packed where those within theirs are the
    larger part of the launch, and not where it is."""
    rng = np.random.default_rng(1)
    lim, z = (0.45, 31) if dt == np.float32 else (0.47, 31)

    def inst(x, y, share, seed):
        return hip.Instance(X=(rng.random((x, y)) < share).astype(dt), z=z, params=hip.Params(1.0, 1.0, [1.0] * x, [1.0] * z),
                            seed=seed)

    def memory(insts, eps=1e-50):
        with hip.Batch(insts, dtype=dt, eps=eps) as b:
            return b.info()["device_bytes"]
    past = inst(100, 90, lim, 0)
    large, small = inst(400, 300, 0.1, 1), inst(60, 50, 0.1, 2)
    extra = [memory(i) - memory(i, 1e-250) for i in ([past], [large], [small], [past, large], [past, small])]
    assert extra[0] == 0 and extra[1] > 0 and extra[2] > 0
    packed_S = 100 * 90 * lim * z * np.dtype(dt).itemsize  # (work lists differ by less)
    assert extra[3] > extra[1] + packed_S
    assert extra[4] < extra[2] + packed_S
