"""The rebuild's fused passes against its definition, cell by cell.

After a cycle one pass does the damage, the water and the removal mask, and in
the FP64 path one more does the properties and the face coefficients, working
out its neighbours' properties by itself.  On grids at the ends of a 256-thread
block and in both thermal modes:
* the fields after a rebuild are those of a plain NumPy restatement
  (setupThermalCoeff as a sequential sweep), to 1e-14 of each value: the same
  FP64 expressions, whose exp and divisions may differ in the last bits;
* a FP64 step after the rebuild, whose faces the fused pass built, matches one
  computed from the downloaded properties, to 1e-12 of the temperature: some 20
  roundings of 1.1e-16 on terms that are at most 10 times the temperature;
* a captured cycle and the same stages called one by one agree bit for bit.
"""
import numpy as np
import pytest

from tam_amd import configs, lib

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (3, 2, 5), (16, 8, 2), (17, 5, 3), (40, 33, 29)]


def _problem(n, water, fp64, seed):
    nx, ny, nz = n
    p = configs._config_params(n, (0.01 * nx, 0.01 * ny, 0.01 * nz))
    p.heat_fp64 = fp64
    p.robin_top = 0
    p.boil = 1 if water else 0
    p.removed_inert = 0 if water else 1
    p.thermal_mode = lib.THERMAL_WATER if water else lib.THERMAL_TABLE
    p.ablate_K = 373.0
    temp, kappa, density, heatcap = configs._thermal_cube(p, configs.C0_THERMAL)
    rng = np.random.default_rng(seed)
    temp = temp.copy()
    temp[1:-1, 1:-1, 1:-1] = 310.0 + 75.0 * rng.random((nz, ny, nx))
    rhokap = np.zeros((nz + 2, ny + 2, nx + 2))
    rhokap[1:-1, 1:-1, 1:-1] = np.where(rng.random((nz, ny, nx)) < 0.3, 0.0, 100.5)
    prob = configs.Problem("passes", p, np.zeros((nz, ny, nx), np.uint8), [(0.5, 100.0, 0.9, 1.38)], temp, kappa,
                           density, heatcap, rhokap=rhokap)
    q = p.qvapor * rng.random((nz, ny, nx))
    return prob, q


def _sweep(T, rk, ablate):
    """the mask as setupThermalCoeff's in-place sweep finds it"""
    rk = rk.copy()
    nz, ny, nx = (s - 2 for s in rk.shape)
    mask = np.zeros((nz, ny, nx), bool)
    for k in range(1, nz + 1):
        for j in range(1, ny + 1):
            for i in range(1, nx + 1):
                empty = (rk[k, j, i + 1] + rk[k, j, i - 1] + rk[k, j + 1, i] + rk[k, j - 1, i] + rk[k + 1, j, i] +
                         rk[k - 1, j, i]) == 0.0
                if T[k, j, i] >= ablate or rk[k, j, i] == 0.0 or empty:
                    mask[k - 1, j - 1, i - 1] = True
                    rk[k, j, i] = 0.0
    return mask


@pytest.mark.parametrize("n", SIZES, ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("water,fp64", [(True, 1), (False, 1), (False, 0)])
def test_rebuild_fields(n, water, fp64):
    prob, q = _problem(n, water, fp64, seed=sum(n))
    p = prob.params
    g = prob.grid()
    if water:
        g.upload(lib.FIELD_Q, q)
    shape = prob.temp.shape
    get = lambda f: g.download(f).reshape(shape)
    T, rk, K, D, H = (get(f) for f in (lib.FIELD_TEMP, lib.FIELD_RHOKAP, lib.FIELD_KAPPA, lib.FIELD_DENSITY,
                                       lib.FIELD_HEATCAP))
    C = get(lib.FIELD_COEFF)
    mask = _sweep(T, rk, p.ablate_K)
    print(n, water, fp64, "removed", int(mask.sum()), flush=True)
    g.rebuild()
    ii = (slice(1, -1),) * 3
    if water:
        W = np.clip(np.minimum(np.minimum(0.75 - 0.75 * (q / p.qvapor), 0.75), 0.75), 0.0, None)
        prot = 1.0 - 0.75
        rho = 1000.0 / (W + 0.649 * prot)
        D[ii] = rho
        H[ii] = 1000.0 * (4.2 * W + 1.09 * prot)
        K[ii] = rho * (6.28e-4 * W + 1.17e-4 * prot)
        rk[ii] = W * p.mu_water + p.mu_protein
        C[ii] = p.delt / (D[ii] * H[ii])
    Ti = T[ii]
    D[ii] = np.where(mask, 101.325e3 / (287.058 * Ti), D[ii])
    H[ii] = np.where(mask, 1.006e3, H[ii])
    K[ii] = np.where(mask, -0.188521 * np.exp(-0.000367259 * (Ti - 273.15)) + 0.212453, K[ii])
    rk[ii] = np.where(mask, 0.0, rk[ii])
    C[ii] = np.where(mask, p.delt / (D[ii] * H[ii]), C[ii])
    for f, want in ((lib.FIELD_RHOKAP, rk), (lib.FIELD_DENSITY, D), (lib.FIELD_HEATCAP, H), (lib.FIELD_COEFF, C)):
        np.testing.assert_allclose(get(f), want, rtol=1e-14, atol=0)
    # the air's conductivity is a difference of two terms near 0.2
    np.testing.assert_allclose(get(lib.FIELD_KAPPA), K, rtol=1e-14, atol=2e-16)
    if fp64 and not p.boil:
        g.heat_run(1)
        K, D, H = get(lib.FIELD_KAPPA), get(lib.FIELD_DENSITY), get(lib.FIELD_HEATCAP)
        gone = np.zeros(shape, bool)
        gone[ii] = get(lib.FIELD_RHOKAP)[ii] == 0.0
        inc = np.zeros(shape)
        for ax, h in ((2, p.dx_m), (1, p.dy_m), (0, p.dz_m)):
            lo = tuple(slice(0, -1) if d == ax else slice(1, -1) for d in range(3))
            hi = tuple(slice(1, None) if d == ax else slice(1, -1) for d in range(3))
            a = p.dscale * ((K[lo] + K[hi]) / 2 / ((D[lo] + D[hi]) / 2 * ((H[lo] + H[hi]) / 2))) / (h * h)
            a = np.where(gone[lo] | gone[hi], 0.0, a) * (T[hi] - T[lo])
            inc[ii] += np.diff(a, axis=ax)
        np.testing.assert_allclose(get(lib.FIELD_TEMP)[ii], T[ii] + p.delt * inc[ii], rtol=1e-12, atol=0)
    g.close()


@pytest.mark.parametrize("water,fp64", [(True, 1), (False, 0)])
def test_cycle_equals_stages(water, fp64):
    n = (17, 12, 9)
    prob, q = _problem(n, water, fp64, seed=3)
    p = prob.params
    p.arr_A, p.arr_dE = 3.1e98, 6.28e5
    p.delt = 2e-5                           # stable beside removed voxels: air conducts 100 times as fast
    fields = (lib.FIELD_TEMP, lib.FIELD_TISSUE, lib.FIELD_THRESTIME, lib.FIELD_RHOKAP, lib.FIELD_WATER,
              lib.FIELD_KAPPA, lib.FIELD_COEFF)
    jm = 1e8 * np.random.default_rng(1).random((n[2], n[1], n[0]))
    outs = []
    for captured in (True, False):
        g = prob.grid()
        g.upload(lib.FIELD_JMEAN, jm)
        t = 0.0
        for c in range(4):
            print("captured" if captured else "stages", c, flush=True)
            if captured:
                g.cycle(0, 1, c, 1.0, 3, arr_delt=3 * p.delt)
            else:
                g.heat_run(3)
                for _ in range(3):          # as the grid's own clock advances
                    t += p.delt
                g.arrhenius(3 * p.delt, t)
                g.rebuild()
        g.synchronize()
        outs.append([g.download(f) for f in fields])
        g.close()
    for a, b in zip(*outs):
        assert np.array_equal(a, b)
