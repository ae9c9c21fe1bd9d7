"""Captured FP64 cycles with packets and several steps: the first step
normalises the run's tally, and the run's counters join the sums.

* jmean is the tally times mu_a times the scale, to the rounding of three
  products (1e-15), and stays for the cycle's further steps and for a cycle
  without packets;
* the counters of several cycles, some asked for and some not, are the sums of
  the same runs made one at a time;
* temperatures and damage agree with the stages called one by one, whose
  tallies differ by the order of FP64 adds (1e-9 of the rise).
"""
import numpy as np
import pytest

from tam_amd import configs, lib

pytestmark = pytest.mark.gpu

COUNTS = ("packets", "absorbed", "specular", "missed", "killed", "crossings", "interactions", "tally_adds", "box_adds")


def _problem(water):
    if water:
        prob = configs.reference_default(n=20)
        prob.params.boil = 0
        return prob, 1e-3 * prob.power
    n = (21, 18, 16)
    p = configs._config_params(n, (0.02 * n[0], 0.02 * n[1], 0.02 * n[2]))
    p.heat_fp64 = 1
    p.robin_top = 0
    p.beam, p.beam_radius = 1, 0.05
    temp, kappa, density, heatcap = configs._thermal_cube(p, configs.C0_THERMAL)
    mat = (np.arange(n[0] * n[1] * n[2]) % 2).astype(np.uint8).reshape(n[::-1])
    prob = configs.Problem("cycles", p, mat, [(0.5, 100.0, 0.9, 1.38), (2.0, 50.0, 0.8, 1.4)], temp, kappa, density,
                           heatcap)
    return prob, 0.05


def _mua_fraction(prob):
    f = np.array([t[0] / (t[0] + t[1]) for t in prob.table])
    return f[prob.mat]


@pytest.mark.parametrize("water", [True, False])
@pytest.mark.parametrize("loops", [1, 2, 3])
def test_captured_cycles_with_packets(water, loops):
    prob, power = _problem(water)
    p = prob.params
    npk, seed = 30_000, 17
    scale = power / (npk * p.volume_voxel)
    a, b = prob.grid(), prob.grid()
    start = a.download(lib.FIELD_TEMP)
    sums, t = np.zeros(len(COUNTS) + 6), 0.0
    for c in range(5):
        print("case", "water" if water else "table", loops, "cycle", c, flush=True)
        # stages
        s = a.mc_run(npk, seed=seed, stream=c)
        a.normalise(scale)
        a.heat_run(loops)
        for _ in range(loops):                       # as the grid's own clock advances
            t += p.delt
        a.arrhenius(loops * p.delt, t)
        a.rebuild()
        sums += [getattr(s, k) for k in COUNTS] + list(s.escaped)
        # one replay; the counters are asked for every other time
        rk = b.download(lib.FIELD_RHOKAP).reshape(start.shape)[1:-1, 1:-1, 1:-1]
        s = b.cycle(npk, seed, c, scale, loops, arr_delt=loops * p.delt, stats=c % 2 == 1)
        if c % 2 == 1:
            assert [getattr(s, k) for k in COUNTS] + list(s.escaped) == sums.tolist()
            sums[:] = 0.0
        tally, jm = b.download(lib.FIELD_TALLY), b.download(lib.FIELD_JMEAN)
        want = tally.reshape(rk.shape) * (rk * _mua_fraction(prob)) * scale
        np.testing.assert_allclose(jm.reshape(rk.shape), want, rtol=1e-15, atol=0)
        assert want.max() > 0
    # without packets: the source stays, and counts nothing
    s = b.cycle(0, seed, 9, scale, loops, arr_delt=loops * p.delt)
    assert [getattr(s, k) for k in COUNTS] + list(s.escaped) == sums.tolist()
    assert np.array_equal(b.download(lib.FIELD_JMEAN), jm)
    a.heat_run(loops)
    for _ in range(loops):
        t += p.delt
    a.arrhenius(loops * p.delt, t)
    a.rebuild()
    Ta, Tb = a.download(lib.FIELD_TEMP), b.download(lib.FIELD_TEMP)
    rise = np.abs(Ta - start).max()
    print("rise", rise, "largest difference", np.abs(Ta - Tb).max(), flush=True)
    assert rise > 0.01
    assert np.abs(Ta - Tb).max() <= 1e-9 * rise + 1e-12 * Ta.max()
    np.testing.assert_allclose(b.download(lib.FIELD_TISSUE), a.download(lib.FIELD_TISSUE), rtol=1e-7, atol=1e-300)
    a.close()
    b.close()
