"""The two-step stencil at the edges of its tiles.

A block owns 30 x 6, 30 x 14 or 62 x 6 columns; lanes on the footprint's edge
fetch the column outside it, the last blocks reach past the grid, and a march
ends at plane nz + 1.  Grids one column or plane to either side of those sizes,
down to one voxel, run the same steps with one step per launch and with two:
fields, Omega and threshold times are bit-identical.  The damage window is the
usual one, one without an upper end, and one without either end.
"""
import numpy as np
import pytest

from tam_amd import configs, lib

pytestmark = pytest.mark.gpu

ONE_STEP = 4                # direct-32x8
EDGES = [(1, 1, 1), (2, 1, 3), (29, 13, 4), (30, 14, 7), (31, 15, 8), (32, 6, 9), (33, 7, 5), (61, 29, 3),
         (62, 28, 2), (63, 5, 17), (65, 16, 1)]
WINDOWS = {"usual": None, "no upper end": (316.0, np.inf), "no end": (-np.inf, 1e30)}


def _block(n, window, seed):
    nx, ny, nz = n
    p = configs._config_params(n, (0.01 * nx, 0.01 * ny, 0.01 * nz))
    p.damage_every_step = 1
    p.arr_A, p.arr_dE = 3.1e98, 6.28e5
    if window:
        p.arr_Tlo, p.arr_Thi = window
    rng = np.random.default_rng(seed)
    temp, kappa, density, heatcap = configs._thermal_cube(p, configs.C0_THERMAL)
    temp = temp.copy()
    temp[1:-1, 1:-1, 1:-1] = 300.0 + 70.0 * rng.random((nz, ny, nx))
    rhokap = np.zeros((nz + 2, ny + 2, nx + 2))
    rhokap[1:-1, 1:-1, 1:-1] = np.where(rng.random((nz, ny, nx)) < 0.1, 0.0, 100.5)     # removed voxels: mixed waves
    mat = np.zeros((nz, ny, nx), np.uint8)
    prob = configs.Problem("edges", p, mat, [(0.5, 100.0, 0.9, 1.38)], temp, kappa, density, heatcap, rhokap=rhokap)
    return prob, 5e7 * rng.random((nz, ny, nx))


def _run(prob, jm, tile, kz, steps):
    g = prob.grid()
    g.upload(lib.FIELD_JMEAN, jm)
    g.set_heat_launch(tile, kz)
    g.heat_run(steps)
    out = [g.download(f) for f in (lib.FIELD_TEMP, lib.FIELD_TISSUE, lib.FIELD_THRESTIME)]
    g.close()
    return out


@pytest.mark.parametrize("window", list(WINDOWS))
@pytest.mark.parametrize("n", EDGES, ids=lambda n: "x".join(map(str, n)))
def test_two_steps_at_tile_edges(n, window):
    prob, jm = _block(n, WINDOWS[window], seed=sum(n))
    want = _run(prob, jm, ONE_STEP, 8, 5)
    assert n == (1, 1, 1) or want[1].any()                  # damage did happen
    for tile, kz in ((6, 1), (6, 4), (7, 2), (7, 8), (8, 3), (8, 32)):
        print(n, window, tile, kz, flush=True)
        got = _run(prob, jm, tile, kz, 5)
        for w, h in zip(want, got):
            assert np.array_equal(w, h)
