"""An FP32 solve of bld_appr does every operation in FP32, whatever the share of
nonempty entries. eps = 1e-50 and 1e-250 are both 0 there, so they cannot tell
two solves apart; in double they lie on both sides of what the lists of nonempty
entries accept (eps of 1e-200 or more)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class _Inst:
    def __init__(self, hip, x, y, z, share, seed):
        rng = np.random.default_rng(seed)
        self.X = ((rng.poisson(2.0, (x, y)) + 1.0) * (rng.random((x, y)) < share)).astype(np.float32)
        self.z, self.seed = z, seed
        self.params = hip.Params(40.0, 1.0, [1.0] * x, [1.0] * z)
        self.nu0 = rng.dirichlet(np.ones(z), size=x).astype(np.float32)
        self.mu0 = rng.dirichlet(np.ones(z), size=y).T.astype(np.float32).copy()


SHAPES = [(8, 10, 3), (33, 65, 7), (200, 150, 32), (300, 40, 17), (150, 200, 64)]


@pytest.mark.parametrize("share", [0.02, 0.2, 1.0])
def test_eps_below_the_range_of_f32(hip, share):
    insts = [_Inst(hip, *s, share, n) for n, s in enumerate(SHAPES)]
    got = []
    for eps in (1e-50, 1e-250):
        with hip.ApprBatch(insts, dtype=np.float32, eps=eps) as b:
            b.solve(15)
            got.append([b.get(n) for n in range(len(insts))])
    for n, (a, b) in enumerate(zip(*got)):
        for u, v in zip(a, b):
            assert np.array_equal(u, v, equal_nan=True), SHAPES[n]
