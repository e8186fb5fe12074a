"""bld_mult in FP64 for instances of one tile (bld_tiny.hip: a whole solve in one
launch) against the step passes, which a batch with a larger instance runs:
equal bit for bit, S and the factors taken from its sums. Shapes: single
elements and rows, full tile rows, z of every lane split and around powers of
two, the most elements it takes and one fiber more; X with empty fibers and with
S + 1 past 10 (the digamma's other branch)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (1, 32, 4), (64, 1, 5), (8, 10, 3), (64, 32, 2), (33, 31, 1), (17, 29, 7), (16, 32, 8), (5, 30, 25),
          (4, 32, 32), (9, 13, 33), (4, 16, 64), (64, 1, 64), (16, 15, 17), (16, 16, 16), (17, 16, 16)]


class _Inst:
    def __init__(self, hip, x, y, z, seed):
        rng = np.random.default_rng(seed)
        self.X = (rng.poisson(3.0, (x, y)) + 1.0) * (rng.random((x, y)) < 0.7)
        self.X[-1, -1] = 17.0
        self.S0 = self.X[:, :, None] * rng.dirichlet(np.full(z, 0.4), size=(x, y))
        self.z, self.seed = z, 1
        self.params = hip.Params(10.0, 1.0, list(rng.uniform(0.5, 2.0, x)), list(rng.uniform(0.8, 2.0, z)))


@pytest.mark.parametrize("appr", [False, True])
def test_tiny_equals_passes(hip, appr):
    small = [_Inst(hip, *s, seed=n) for n, s in enumerate(SHAPES)]
    large = _Inst(hip, 130, 70, 5, 99)
    with hip.Batch(small + [large], dtype=np.float64, use_psi_appr=appr) as passes:
        for iters in (1, 2, 11):
            passes.solve(iters)
            for n, i in enumerate(small):
                with hip.Batch([i], dtype=np.float64, use_psi_appr=appr) as alone:
                    alone.solve(iters)
                    S = alone.S(0)
                    # a single row's gradients cancel (0 / 0 in the reference too)
                    assert SHAPES[n][0] == 1 or (np.all(np.isfinite(S)) and S.any())
                    assert np.array_equal(S, passes.S(n), equal_nan=True), (SHAPES[n], iters)
                    for a, b in zip(alone.fact(0), passes.fact(n)):
                        assert np.array_equal(a, b, equal_nan=True), (SHAPES[n], iters)


def test_tiny_continues_a_solve(hip):
    """Checked every 3 iterations, solved in one go, and among others."""
    insts = [_Inst(hip, *s, seed=n) for n, s in enumerate(SHAPES)]
    with hip.Batch(insts, dtype=np.float64) as b:
        b.solve(10)
        ref = [b.S(n) for n in range(len(insts))]
        ran, _ = b.solve_tol(10, 0.0, 3)
        assert ran == 10
        for n, r in enumerate(ref):
            assert np.array_equal(b.S(n), r, equal_nan=True), SHAPES[n]
