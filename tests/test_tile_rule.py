"""Heights of small FP64 instances' tiles: about 5120 elements, at least 8 rows
(rounded to a multiple of 4 of equal tiles), at most 1024 tiles; FP32 and the
instances of 2^20 fibers or more keep theirs."""
import numpy as np
import pytest


@pytest.mark.parametrize("shape,f64,f32", [((100, 100, 17), 8, 52), ((8, 10, 3), 8, 8), ((384, 300, 32), 8, 64),
                                           ((256, 128, 64), 8, 64), ((50, 60, 8), 20, 52), ((3, 5, 64), 4, 4),
                                           ((1000, 10, 8), 64, 64), ((1, 70, 33), 4, 4), ((900, 1100, 20), 32, 60)])
def test_heights(hip, shape, f64, f32):
    x, y, z = shape
    old = [hip.tune_get(dt, z, x * y) for dt in (np.float64, np.float32)]
    try:
        for dt in (np.float64, np.float32):
            hip.tune_set(dt, z, x * y, 0)
        assert hip.tile_rows(np.float64, x, y, z) == f64
        assert hip.tile_rows(np.float32, x, y, z) == f32
    finally:
        for dt, rows in zip((np.float64, np.float32), old):
            hip.tune_set(dt, z, x * y, rows)
