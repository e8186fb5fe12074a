"""Fibers of 65 to 256 elements in registers (bld_wide.hip): every register
count, its last fully and barely used lane, ragged and single-fiber tiles, for
the multiplicative and the additive step, against the oracle. FP64 bound 1e-10
relative normwise and FP32 (x >= 40) 1e-4, as for the other deep fibers.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 65), (3, 40, 128), (17, 15, 129), (16, 16, 192), (15, 33, 193), (18, 7, 256)]
SHAPES32 = [(40, 17, 65), (41, 31, 128), (49, 16, 129), (40, 9, 192), (47, 18, 193), (48, 20, 256)]


def _rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    nb = np.linalg.norm(b)
    return float(np.linalg.norm(a - b) / nb) if nb > 0 else float(np.linalg.norm(a))


@pytest.mark.parametrize("shape", SHAPES)
def test_fp64(hip, oracle, shape):
    x, y, z = shape
    p = hip.Params(40.0, 1.0, [1.0] * x, [1.0] * z)
    X = hip.sample_X(z + y, (x, y, z), p)
    S0 = hip.init_S(z, X, z)
    for appr in (False, True):
        got = hip.bld_mult(X, z, p, 8, appr, S0=S0)
        assert _rel(got, oracle.bld_mult(X, z, p.alpha, p.beta, S0, max_iter=8, use_psi_appr=appr)) <= 1e-10, appr
    got = hip.bld_add(X, z, p, 8, S0=S0)
    assert _rel(got, oracle.bld_add(X, z, p.alpha, p.beta, S0, max_iter=8)) <= 1e-10


@pytest.mark.parametrize("shape", SHAPES32)
def test_fp32(hip, oracle, shape):
    x, y, z = shape
    p = hip.Params(40.0, 1.0, [1.0] * x, [1.0] * z)
    X = hip.sample_X(z + y, (x, y, z), p)
    S0 = hip.init_S(z, X, z).astype(np.float32)
    got = hip.bld_mult(X.astype(np.float32), z, p, 8, True, S0=S0, dtype=np.float32)
    ref = oracle.bld_mult(X, z, p.alpha, p.beta, S0.astype(np.float64), max_iter=8, use_psi_appr=True)
    assert _rel(got, ref) <= 1e-4
    got = hip.bld_add(X.astype(np.float32), z, p, 8, S0=S0, dtype=np.float32)
    assert _rel(got, oracle.bld_add(X, z, p.alpha, p.beta, S0.astype(np.float64), max_iter=8)) <= 1e-4
