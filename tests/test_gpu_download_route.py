"""Field downloads at the sizes where the way to host memory changes: each
value is exact with no ring idle (a plain copy) and with one."""
import numpy as np
import pytest

from tam_amd import configs, lib

pytestmark = pytest.mark.gpu


# results just below, at and above 16 KiB, 160 KiB and 2 MiB
@pytest.mark.parametrize("n", [1, 2047, 2048, 2049, 20478, 20480, 20482, 262143, 262144, 262145])
@pytest.mark.parametrize("idle", [False, True])
def test_values_at_the_lines(n, idle):
    print("case", n, "idle ring" if idle else "no ring", flush=True)
    fx = next(f for f in range(4096, 0, -1) if n % f == 0 and n // f <= 4096)
    shape = (1, n // fx, fx)
    p = configs._config_params(shape[::-1], tuple(0.01 * s for s in shape[::-1]))
    temp, kappa, density, heatcap = configs._thermal_cube(p, configs.C0_THERMAL)
    rng = np.random.default_rng(n)
    temp = 300.0 + 60.0 * rng.random(temp.shape)
    mat = rng.integers(0, 2, shape).astype(np.uint8)
    prob = configs.Problem("download", p, mat, [(0.5, 100.0, 0.9, 1.38), (0.7, 69.3, 0.9, 1.38)], temp, kappa, density,
                           heatcap)
    g = prob.grid()
    jm = rng.random(shape)
    g.upload(lib.FIELD_JMEAN, jm)
    if idle:
        big = configs.config0(n=80).grid()                   # 4 MB: makes a ring and leaves it idle
        big.download(lib.FIELD_TALLY)
    for _ in range(2):
        assert np.array_equal(g.download(lib.FIELD_JMEAN), jm)
        assert np.array_equal(g.download(lib.FIELD_MAT), mat.astype(float))
        want = p.t_ref + (temp - p.t_ref).astype(np.float32).astype(np.float64)
        assert np.array_equal(g.download(lib.FIELD_TEMP), want)
        assert not g.download(lib.FIELD_THRESTIME).any()
    g.close()
    if idle:
        big.close()
