"""The approximate solver over the nonempty entries of X (bld_appr_live.hip)
against the oracle, on both sides of the rule that chooses it: shares of nonempty entries from almost none to all, empty rows and columns, lists for one
and for four wavefronts, z at and around powers of two.

FP64 bounds are those of tests/test_gpu_bld_appr.py (1e-12 relative normwise
after one iteration, 1e-10 after twelve). FP32, with roundings of
2^-24 = 6e-8 and psi good to a few 1e-7 against gradients of order 1: 1e-5; there factors
that turned negative are left out, since FP32's psi(S + 1) is for S >= 0.
bld_appr's factors may change sign, and its trajectory is then chaotic: an
instance is not compared where the oracle's own answer moves by more than 1e-13
(FP32: 1e-6) when its start is moved in the last bit. Alone and batched agree
bitwise everywhere.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (5, 3, 2), (4, 260, 3), (300, 5, 4), (33, 65, 7), (64, 63, 8), (90, 40, 17), (40, 41, 32), (30, 50, 33),
          (70, 20, 64), (20, 30, 65)]
SHARES = [0.03, 0.2, 0.5, 0.95, 1.0]


class _Inst:
    def __init__(self, X, z, params, nu0, mu0):
        self.X, self.z, self.params, self.nu0, self.mu0, self.seed = X, z, params, nu0, mu0, 0


def _problem(hip, shape, share, seed, dtype):
    x, y, z = shape
    rng = np.random.default_rng(seed)
    X = (rng.poisson(2.0, (x, y)) + 1.0) * (rng.random((x, y)) < share)
    if x > 2 and y > 2 and share < 1:
        X[1] = 0
        X[:, y - 2] = 0
    p = hip.Params(40.0, 1.0, list(rng.uniform(0.2, 2.0, x)), list(rng.uniform(0.2, 2.0, z)))
    nu0 = rng.dirichlet(np.ones(z), size=x).astype(dtype)
    mu0 = rng.dirichlet(np.ones(z), size=y).T.astype(dtype).copy()
    return _Inst(X.astype(dtype), z, p, nu0, mu0)


def _rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    nb = np.linalg.norm(b)
    return np.linalg.norm(a - b) / nb if nb > 0 else np.linalg.norm(a)


def _oracle(oracle, i, iters, dtype):
    """The oracle's S, nu, mu, and how far they move with the start's last bit."""
    def run(ulp):
        s = np.random.default_rng(5).choice([-ulp, ulp], i.nu0.size + i.mu0.size)
        nu0 = i.nu0.astype(np.float64) * (1 + s[:i.nu0.size].reshape(i.nu0.shape))
        mu0 = i.mu0.astype(np.float64) * (1 + s[i.nu0.size:].reshape(i.mu0.shape))
        return oracle.bld_appr(i.X.astype(np.float64), i.z, i.params.alpha, i.params.beta, nu0, mu0, max_iter=iters)
    ref = run(0.0)
    return ref, np.max([_rel(a, b) for a, b in zip(run(np.finfo(dtype).eps / 2), ref)])


@pytest.mark.parametrize("share", SHARES)
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_appr_over_nonempty_entries(hip, oracle, dtype, share):
    insts = [_problem(hip, s, share, 11 * n + 1, dtype) for n, s in enumerate(SHAPES)]
    compared = 0
    with hip.ApprBatch(insts, dtype=dtype) as b:
        for iters in (12, 1):
            tol = 1e-5 if dtype == np.float32 else (1e-12 if iters == 1 else 1e-10)
            b.solve(iters)
            for n, i in enumerate(insts):
                got = b.get(n)
                ref, moves = _oracle(oracle, i, iters, dtype)
                steady = moves < (1e-6 if dtype == np.float32 else 1e-13)
                if dtype == np.float32 and min(ref[1].min(), ref[2].min()) < 0:
                    steady = False
                compared += steady
                for g, r, what in zip(got, ref, ("S", "nu", "mu")):
                    assert not steady or _rel(g, r) < tol, (SHAPES[n], share, iters, what, _rel(g, r))
                alone = hip.bld_appr(i.X, i.z, i.params, iters, nu0=i.nu0, mu0=i.mu0, dtype=dtype)
                for g, a in zip(got, alone):
                    assert np.array_equal(g, a, equal_nan=True), (SHAPES[n], share, iters)
    assert compared >= len(SHAPES)


@pytest.mark.parametrize("n", range(len(SHAPES) - 1))
def test_appr_f32_iterates_in_double(hip, oracle, n):
    """An FP32 instance over lists is solved in double from its FP32 start: nu and
    mu carry one rounding (2^-24 = 6e-8; 1e-7 with the FP64 bound), S the roundings
    of an FP32 sum of z products and five more operations, (z + 5) 2^-24 at most."""
    i = _problem(hip, SHAPES[n], 0.03, 11 * n + 1, np.float32)
    ref, moves = _oracle(oracle, i, 12, np.float64)
    S, nu, mu = hip.bld_appr(i.X, i.z, i.params, 12, nu0=i.nu0, mu0=i.mu0, dtype=np.float32)
    if not moves < 1e-13:
        return  # no trajectory to compare, see above
    assert _rel(nu, ref[1]) < 1e-7 and _rel(mu, ref[2]) < 1e-7
    assert _rel(S, ref[0]) < (i.z + 5) * 2.0 ** -24 + 1e-10
