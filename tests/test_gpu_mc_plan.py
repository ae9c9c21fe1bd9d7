"""The LDS box of a transport run on the device: it is its launch shape's, whether
the packets justify all of the shape's blocks or fewer, in the runs and in the
tuner's samples; and the material tables beside it."""
import numpy as np
import pytest

from tam_amd import configs, lib

pytestmark = pytest.mark.gpu

ONE, TWO, THREE, SIX = (42, 42, 46), (34, 34, 34), (28, 28, 34), (22, 22, 27)     # boxes by blocks a CU


def _grid():
    return configs.three_layer_skin(n=(64, 64, 64), ext=(0.5, 0.5, 0.25), packets=1, steps=1).grid()


@pytest.mark.parametrize("shape,packets,box", [(8, 200_000, TWO), (8, 1_000_000, TWO), (6, 1_000_000, SIX),
                                               (4, 1_000_000, ONE), (3, 1_000_000, THREE), (2, 1_000_000, TWO),
                                               (8, 8_388_608, TWO)])
def test_box_of_the_shape(shape, packets, box):
    print("case", shape, packets, box, flush=True)
    g = _grid()
    g.set_mc_box(False)
    g.set_mc_launch(shape, 32)
    a = g.mc_run(packets, seed=11)
    ta = g.download(lib.FIELD_TALLY)
    g.set_mc_box(True, fp64=False)
    b = g.mc_run(packets, seed=11)
    tb = g.download(lib.FIELD_TALLY)
    assert g.mc_box()[1] == box
    assert b.box_adds > 0
    for k in ("absorbed", "specular", "missed", "killed", "crossings", "interactions", "tally_adds"):
        assert getattr(a, k) == getattr(b, k), k
    assert list(a.escaped) == list(b.escaped)
    # each deposit rounded to 2^-13 of dx + dy + dz, half a unit at most: relative to a voxel's deposits,
    # of a few hundredths of that length on average, below 1e-3, and single ones by a few units
    unit = (0.5 / 64 + 0.5 / 64 + 0.25 / 64) / 2 ** 13
    np.testing.assert_allclose(tb, ta, rtol=1e-3, atol=16 * unit)
    g.close()


def test_the_tuner_launches_all_blocks_of_a_shape():
    print("case: tuning on 1e6 packets; its last launch is 8 blocks a CU with the box", flush=True)
    g = _grid()
    g.tune_mc(1_000_000)
    assert g.mc_box()[1] == TWO
    g.close()


# the table behind the largest box: 15 materials and air are 16 entries, the
# most that fit below the box's own 1 KiB; 28 entries the most that fit at all
@pytest.mark.parametrize("materials", [15, 16, 27, 28, 63, 64])
def test_material_tables_at_the_lds_limit(materials):
    print("case: materials", materials, flush=True)
    prob = configs.three_layer_skin(n=(64, 64, 64), ext=(0.5, 0.5, 0.25), packets=1, steps=1)
    prob.table = [(2.0 + 0.1 * m, 150.0 + m, 0.8, 1.4) for m in range(materials)]
    prob.mat = (np.arange(prob.mat.size) % materials).astype(np.uint8).reshape(prob.mat.shape)
    a, b = prob.grid(), prob.grid()
    b.upload(lib.FIELD_RHOKAP, b.download(lib.FIELD_RHOKAP))          # mu_t from the array
    for shape, box in ((4, True), (1, True), (4, False)):
        for g in (a, b):
            g.set_mc_launch(shape, 32)
            g.set_mc_box(box)
        sa, sb = (g.mc_run(300_000, seed=4) for g in (a, b))
        assert not box or a.mc_box()[1] == ONE
        for k in ("absorbed", "specular", "missed", "killed", "crossings", "interactions", "tally_adds", "box_adds"):
            assert getattr(sa, k) == getattr(sb, k), k
        assert list(sa.escaped) == list(sb.escaped)
        ta, tb = (g.download(lib.FIELD_TALLY) for g in (a, b))
        np.testing.assert_allclose(ta, tb, rtol=1e-9, atol=1e-9 * tb.max())
    a.close()
    b.close()


# a batched wave's table holds 4 entries, air included; past that mu_t comes from the array
@pytest.mark.parametrize("materials", [3, 4, 9])
@pytest.mark.parametrize("shape", [3, 4])
def test_batched_tissues_of_several_materials(materials, shape):
    print("case: batch,", materials, "materials,", shape, "blocks a CU", flush=True)
    probs = []
    for q, n in enumerate(((33, 28, 40), (48, 48, 48), (20, 61, 17))):
        prob = configs.three_layer_skin(n=n, ext=(0.5, 0.5, 0.25), packets=1, steps=1)
        prob.table = [(2.0 + 0.3 * m, 90.0 + 5.0 * q + m, 0.8, 1.4) for m in range(materials)]
        prob.mat = (np.arange(prob.mat.size) % materials).astype(np.uint8).reshape(prob.mat.shape)
        prob.params.damage_every_step = 0
        probs.append(prob)
    gs = [p.grid() for p in probs]
    b = lib.Batch(gs)
    b.set_launch(4, 8, shape, 32)
    npk = [60_000, 150_000, 40_000]
    st = b.mc_run(npk, seed=6, stream0=2)
    tb = [g.download(lib.FIELD_TALLY) for g in gs]
    b.close()
    for i, g in enumerate(gs):
        g.set_mc_launch(8, 32)
        g.set_mc_box(False)
        s1 = g.mc_run(npk[i], seed=6, stream=2 + i)
        t1 = g.download(lib.FIELD_TALLY)
        for k in ("absorbed", "specular", "missed", "killed", "crossings", "interactions", "tally_adds"):
            assert getattr(st[i], k) == getattr(s1, k), (i, k)
        assert list(st[i].escaped) == list(s1.escaped)
        p = probs[i].params
        # deposits rounded to the box's unit, half a unit each: as for one material (test_gpu_batch)
        unit = 2.0 * (p.xmax / p.nx + p.ymax / p.ny + p.zmax / p.nz) / 2 ** 13
        np.testing.assert_allclose(tb[i], t1, rtol=1e-4, atol=16 * unit)
        g.close()


def test_batched_grids_one_voxel_wide():
    """Without a box: a word of the 16-bit box holds two x neighbours, and its
    carry goes to the second."""
    sizes = [(1, 20, 33), (24, 1, 40), (1, 1, 61), (30, 30, 30)]
    print("case: batch of", sizes, flush=True)
    probs = []
    for n in sizes:
        prob = configs.three_layer_skin(n=n, ext=(0.2, 0.2, 0.5), packets=1, steps=1)
        prob.params.damage_every_step = 0
        probs.append(prob)
    gs = [p.grid() for p in probs]
    b = lib.Batch(gs)
    npk = [40_000, 30_000, 50_000, 20_000]
    st = b.mc_run(npk, seed=6, stream0=2)
    tb = [g.download(lib.FIELD_TALLY) for g in gs]
    b.close()
    for i, g in enumerate(gs):
        assert (st[i].box_adds > 0) == (min(sizes[i][:2]) > 1)
        g.set_mc_box(False)
        s1 = g.mc_run(npk[i], seed=6, stream=2 + i)
        t1 = g.download(lib.FIELD_TALLY)
        for k in ("absorbed", "specular", "missed", "killed", "crossings", "interactions", "tally_adds"):
            assert getattr(st[i], k) == getattr(s1, k), (i, k)
        if min(sizes[i][:2]) == 1:
            np.testing.assert_allclose(tb[i], t1, rtol=1e-9, atol=1e-9 * t1.max())
        g.close()
