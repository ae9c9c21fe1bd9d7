"""The transport's launch plan (host arithmetic, CPU only): a run's blocks are
chosen in waves per CU whatever the block size, and the LDS box is the launch
shape's whatever the packets."""
import ctypes as C
import random

import pytest

from tam_amd import lib

NCU, LDS = 256, 160 * 1024
FIELDS = ("box", "lanes", "per_cu", "blocks", "sd", "d", "ntab", "tab_off", "lds", "limit")


def plan(npk, n=(200, 200, 200), shape=8, box=1, nmat=4, by_mat=1, full=0, ncu=NCU, lds_cu=LDS, lds_blk=LDS):
    i64 = C.c_int64
    out = (i64 * len(FIELDS))()
    lib.load().tam_internal_mc_plan((i64 * 12)(npk, *n, shape, box, nmat, by_mat, full, ncu, lds_cu, lds_blk), out)
    return dict(zip(FIELDS, out))


def waves(p):
    """Waves a CU, over the whole device."""
    return p["blocks"] * (p["lanes"] // 64) / NCU


@pytest.mark.parametrize("shape", [1, 2, 3, 4, 5, 6, 7, 8, 12, 16, 64])
@pytest.mark.parametrize("packets", [130_000, 300_000, 1_000_000, 3_000_000, 6_300_000, 8_400_000, 20_000_000, 10 ** 8])
def test_short_box_runs_keep_sixteen_waves_a_cu(shape, packets):
    p = plan(packets, shape=shape)
    few = packets < 64 * NCU * shape
    assert p["box"] == (0 if few else 1)
    if few:
        return
    assert waves(p) >= min(16, 4 * shape)                       # the shape's own where it is smaller
    assert waves(p) <= 4 * shape
    if packets >= 4096 * NCU * shape:                           # 1024 packets for each wave of the shape
        assert waves(p) == 4 * shape
    assert waves(p) <= max(16, packets / (1024 * NCU))
    # the box is the shape's, and so is what is rounded to its units
    assert {k: p[k] for k in ("lanes", "per_cu", "sd", "d", "ntab", "lds")} == \
        {k: plan(10 ** 9, shape=shape)[k] for k in ("lanes", "per_cu", "sd", "d", "ntab", "lds")}
    share = LDS // p["per_cu"] - 1024
    assert p["sd"] == int((share // 2) ** (1 / 3)) & ~1
    assert 2 * p["sd"] ** 2 * (p["d"] + 1) > share >= 2 * p["sd"] ** 2 * p["d"]


@pytest.mark.parametrize("shape", [1, 2, 3, 4, 6, 8])
def test_tuner_samples_run_the_whole_shape(shape):
    long_run = plan(10 ** 8, shape=shape)
    for packets in (2_000_000, 5_000_000):
        assert plan(packets, shape=shape, full=1) == long_run


@pytest.mark.parametrize("shape", [1, 2, 3, 4, 6, 8, 16])
@pytest.mark.parametrize("packets", [1, 4097, 20_000, 140_000, 400_000, 1_000_000, 3_000_000, 8_400_000, 20_000_000, 10 ** 8])
def test_runs_without_the_box_keep_sixteen_waves_a_cu(shape, packets):
    p = plan(packets, shape=shape, box=0)
    assert (p["box"], p["lanes"]) == (0, 256)
    most = 4 * shape
    assert waves(p) <= min(most, max(16, packets / (1024 * NCU))) + 4 / NCU
    assert waves(p) >= min(most, max(min(16, packets / (64 * NCU)), min(8, packets / (4 * NCU)), packets // 1024 / NCU))
    # the tuner's samples stand for longer runs
    assert plan(packets, shape=shape, box=0, full=1)["blocks"] == NCU * shape


def test_box_leaves_the_lds_that_its_blocks_need():
    rng = random.Random(5)
    for _ in range(4000):
        q = dict(npk=int(10 ** rng.uniform(0, 9)), n=tuple(rng.randint(1, 300) for _ in range(3)),
                 shape=rng.randint(1, 64), box=rng.randint(0, 2), nmat=rng.randint(2, 256), by_mat=rng.randint(0, 1),
                 full=rng.randint(0, 1))
        p = plan(**q)
        assert p["blocks"] >= 1 and p["lanes"] in (256, 1024), q
        if not p["box"]:
            assert p["lds"] == 32 * p["ntab"] <= 32 * 64 and waves(p) <= 4 * q["shape"], q
            continue
        esz = 2 if q["box"] == 1 else 8
        bytes_ = esz * p["sd"] ** 2 * p["d"]
        assert p["sd"] <= min(q["n"][:2]) and p["d"] <= q["n"][2], q
        assert bytes_ <= LDS // p["per_cu"] - 1024, q
        assert p["ntab"] in (0, q["nmat"]) and (q["by_mat"] or not p["ntab"]), q
        if p["ntab"]:
            assert p["tab_off"] % 16 == 0 and p["tab_off"] >= bytes_ and p["lds"] == p["tab_off"] + 32 * p["ntab"], q


COUNTS = 14 * 8                                                 # a block's static LDS: its counts


@pytest.mark.parametrize("entries", [2, 16, 17, 28, 29, 64, 256])
def test_box_and_table_fit_what_the_kernel_is_allowed(entries):
    p = plan(10 ** 7, n=(64, 64, 64), shape=4, nmat=entries)
    assert (p["sd"], p["sd"], p["d"]) == (42, 42, 46) and p["ntab"] == (entries if entries <= 28 else 0)
    assert p["lds"] <= p["limit"] == LDS - COUNTS


def test_no_plan_asks_for_more_lds_than_is_allowed():
    rng = random.Random(9)
    for _ in range(4000):
        q = dict(npk=10 ** 9, n=tuple(rng.randint(4, 300) for _ in range(3)), shape=rng.choice([1, 2, 3, 4, 5, 8, 12]),
                 box=rng.randint(1, 2), nmat=rng.randint(2, 64))
        p = plan(**q)
        assert p["lds"] <= p["limit"], q
        if p["ntab"]:                                           # and every block a CU finds its place
            step = LDS // 128
            assert -(-(p["lds"] + COUNTS) // step) * step * p["per_cu"] <= LDS, q


def batch_slots(grids, shape):
    """(slots a wave asks for, each grid's cube)"""
    n = len(grids)
    edges, cube = (C.c_int32 * (3 * n))(*[e for g in grids for e in g]), (C.c_int32 * (2 * n))()
    slots = lib.load().tam_internal_batch_slots(edges, n, NCU, LDS, LDS, shape, cube)
    return slots, [tuple(cube[2 * i:2 * i + 2]) for i in range(n)]


@pytest.mark.parametrize("shape", range(1, 65))
def test_batched_cubes_fit_their_slices(shape):
    rng = random.Random(shape)
    most = min(LDS - 1024, LDS // shape - 1024) // 8 & ~7 if LDS // shape > 1024 else 0
    for _ in range(50):
        grids = [tuple(rng.randint(1, 200) for _ in range(3)) for _ in range(rng.randint(1, 6))]
        slots, cubes = batch_slots(grids, shape)
        assert slots % 8 == 0 and slots <= most
        for (nx, ny, nz), (sd, d) in zip(grids, cubes):
            assert sd % 2 == 0 and sd * sd * d <= slots and sd <= min(nx, ny) and d <= nz
            if sd == 0:                                         # no pair of x neighbours for a word's two slots
                assert min(nx, ny) == 1 or most < 8
                continue
            # the largest: neither edge could be longer
            assert d == nz or sd * sd * (d + 1) > most
            assert sd >= min(nx, ny) - 1 or (sd + 2) ** 3 > most
        assert slots == -(-max(sd * sd * d for sd, d in cubes) // 8) * 8


@pytest.mark.parametrize("shape", [1, 2, 3, 4, 8])
def test_batched_blocks_of_a_cu_find_their_lds(shape):
    """Cubes of ordinary tissues leave the counts and tables of every block of a CU their LDS."""
    slots, _ = batch_slots([(64, 64, 64), (96, 96, 96), (160, 160, 160)], shape)
    static, step = 4 * (COUNTS + 4 * 32), LDS // 128            # a wave's counts and four materials, four times
    block = static + 4 * 2 * slots
    assert block <= LDS and -(-block // step) * step * shape <= LDS


@pytest.mark.parametrize("w", [4, 1024, 4096, 8192])
@pytest.mark.parametrize("packets", [1, 70_000, 300_000, 1_000_000, 3_000_000, 10 ** 7, 3 * 10 ** 7, 10 ** 8, 10 ** 9])
def test_queue_draws_stay_few_and_end_small(w, packets):
    """The draws of all waves are one chain on one address.  A draw of 64 k
    packets is made while 128 w k to 128 w (k + 1) are left (to 0 for k = 1):
    4 w draws of 64 and 2 w / k of each further size up to 256, which is
    never 3.7 w more than draws of 256 would be."""
    last = C.c_int64()
    f = lib.load().tam_internal_mc_draws
    f.restype = C.c_int64
    n = f(C.c_int64(packets), C.c_int64(w), C.byref(last))
    left = max(0, packets - w * min(64, -(-packets // w)))
    assert (n == 0) == (left == 0) and n <= -(-left // 64)
    if left:
        assert last.value == 64
        assert n <= -(-left // 256) + 3.7 * w + 1
