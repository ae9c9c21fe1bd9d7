"""Energy bookkeeping of the FP64 step and of the heat-content sum.

The FP64 step adds each block's boundary outflow to the block's own slot, and
the heat content is summed by a bounded grid that strides over the voxels.
Without a source the content lost is the outflow.  Bound: a step rounds a
temperature by 2^-53 of its absolute value, a sum over a tree or a stride of
at most a few hundred terms by as many roundings of its partial sums, so the
balance and the sum hold to 1e-13 of the sum of rho c V T over absolute T.
"""
import numpy as np
import pytest

from tam_amd import configs, lib

pytestmark = pytest.mark.gpu


# one voxel; less than a block; a block's end; past 2048 blocks of 256 voxels
@pytest.mark.parametrize("n", [(1, 1, 1), (5, 7, 3), (16, 16, 1), (257, 1, 2), (101, 79, 67)])
@pytest.mark.parametrize("fp64", [1, 0])
def test_energy_balance(n, fp64):
    nx, ny, nz = n
    p = configs._config_params(n, (0.01 * nx, 0.01 * ny, 0.01 * nz))
    p.heat_fp64 = fp64
    p.robin_top = 0
    temp, kappa, density, heatcap = configs._thermal_cube(p, configs.C0_THERMAL)
    rng = np.random.default_rng(nx)
    temp = temp.copy()
    temp[1:-1, 1:-1, 1:-1] += 60.0 * rng.random((nz, ny, nx))
    rhokap = np.zeros((nz + 2, ny + 2, nx + 2))
    rhokap[1:-1, 1:-1, 1:-1] = 100.5
    g = configs.Problem("slots", p, np.zeros((nz, ny, nx), np.uint8), [(0.5, 100.0, 0.9, 1.38)], temp, kappa, density,
                        heatcap, rhokap=rhokap).grid()
    cap = heatcap[1:-1, 1:-1, 1:-1] * p.mass_voxel
    before, out0 = g.energy()
    T = g.download(lib.FIELD_TEMP).reshape(temp.shape)[1:-1, 1:-1, 1:-1]
    bound = 1e-13 * float((cap * T).sum())
    print(n, fp64, before, flush=True)
    assert out0 == 0.0
    assert abs(before - float((cap * (T - p.t_ref)).sum())) <= bound
    if fp64:
        g.heat_run(3)
        after, out = g.energy()
        print("lost", before - after, "out", out, "bound", bound, flush=True)
        assert out > 0.0
        assert abs((before - after) - out) <= bound
    g.close()
