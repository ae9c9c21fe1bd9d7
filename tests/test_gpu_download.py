"""Field downloads through the pinned ring.

Sizes around a slot (2 MiB of doubles) and around a ring of eight, to arrays
that start at, before and after a huge page, from several threads at once and
after every context has closed.  A download is a copy (or a conversion in
FP64), so each value is exact.
"""
import ctypes
import threading

import numpy as np
import pytest

from tam_amd import configs, lib

pytestmark = pytest.mark.gpu

SLOT = (2 << 20) // 8


def _grid(n, fp64=0):
    nx, ny, nz = n
    p = configs._config_params(n, (0.01 * nx, 0.01 * ny, 0.01 * nz))
    p.heat_fp64 = fp64
    temp, kappa, density, heatcap = configs._thermal_cube(p, configs.C0_THERMAL)
    rng = np.random.default_rng(nx)
    temp = 300.0 + 60.0 * rng.random(temp.shape)
    mat = rng.integers(0, 2, (nz, ny, nx)).astype(np.uint8)
    rhokap = np.zeros((nz + 2, ny + 2, nx + 2))
    rhokap[1:-1, 1:-1, 1:-1] = np.array([100.5, 70.0])[mat]
    prob = configs.Problem("download", p, mat, [(0.5, 100.0, 0.9, 1.38), (0.7, 69.3, 0.9, 1.38)], temp, kappa, density,
                           heatcap, rhokap=rhokap)
    return prob.grid(), p, temp, mat, rng.random((nz, ny, nx))


# voxels: 1; one slot less one, one slot, one more; eight slots less one and more (8 * 2^18 = 2^21)
SIZES = [(1, 1, 1), (511, 513, 1), (512, 512, 1), (481, 109, 5), (2047, 1025, 1), (128, 128, 129)]


@pytest.mark.parametrize("n", SIZES, ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("fp64", [0, 1])
def test_values(n, fp64):
    print(n, fp64, flush=True)
    g, p, temp, mat, jm = _grid(n, fp64)
    g.upload(lib.FIELD_JMEAN, jm)
    assert np.array_equal(g.download(lib.FIELD_JMEAN).ravel(), jm.ravel())
    assert np.array_equal(g.download(lib.FIELD_MAT).ravel(), mat.ravel().astype(float))
    want = temp if fp64 else p.t_ref + (temp - p.t_ref).astype(np.float32).astype(np.float64)
    assert np.array_equal(g.download(lib.FIELD_TEMP).ravel(), want.ravel())
    assert g.download(lib.FIELD_THRESTIME).size == 3 * jm.size
    g.close()


@pytest.mark.parametrize("shift", [0, 1, SLOT - 1])
def test_destination_alignment(shift):
    g, p, temp, mat, jm = _grid((481, 109, 5))
    g.upload(lib.FIELD_JMEAN, jm)
    buf = np.full(jm.size + 2 * SLOT + 2, -1.0)
    at = (-buf.ctypes.data // 8) % SLOT + shift + 1           # doubles from a huge page, never the first of buf
    out = buf[at:at + jm.size]
    print("address", out.ctypes.data % (2 << 20), flush=True)
    g._chk(g.L.tam_download(g.h, lib.FIELD_JMEAN, out.ctypes.data_as(ctypes.POINTER(ctypes.c_double))))
    assert np.array_equal(out, jm.ravel())
    assert buf[at - 1] == -1.0 and buf[at + jm.size] == -1.0   # nothing beside it is written
    g.close()


def test_threads_and_last_context():
    grids = [_grid((300, 200, 9 + q)) for q in range(4)]
    for g, _, _, _, jm in grids:
        g.upload(lib.FIELD_JMEAN, jm)
    bad = []

    def loop(g, jm):
        for _ in range(5):
            if not np.array_equal(g.download(lib.FIELD_JMEAN).ravel(), jm.ravel()):
                bad.append(1)

    th = [threading.Thread(target=loop, args=(g, jm)) for g, _, _, _, jm in grids]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
    for g, *_ in grids:                                        # the idle rings go with the last one
        g.close()
    g, _, _, _, jm = _grid((300, 200, 9))
    g.upload(lib.FIELD_JMEAN, jm)
    assert np.array_equal(g.download(lib.FIELD_JMEAN).ravel(), jm.ravel())
    g.close()
