"""The march depths that the stencil tuner times (host arithmetic, CPU only):
chosen by the blocks that a launch shape gets on the grid, not by its voxels."""
import ctypes as C
import random

import pytest

from tam_amd import lib

NCU = 256
DIMS = {3: (64, 4), 4: (32, 8), 5: (64, 8), 6: (30, 6), 7: (30, 14), 8: (62, 6)}     # columns a block owns


def depths(tile, n, ncu=NCU):
    out = (C.c_int * 16)()
    k = lib.load().tam_internal_heat_depths(tile, *n, ncu, out)
    return list(out[:k])


def blocks(tile, n, kz):
    tx, ty = DIMS[tile]
    return -(-n[0] // tx) * -(-n[1] // ty) * -(-n[2] // kz)


GRIDS = [(1, 1, 1), (50, 50, 50), (80, 80, 80), (113, 97, 101), (119, 119, 119), (120, 120, 120), (200, 200, 200),
         (32, 32, 1600), (40, 40, 1040), (16, 16, 4096), (4096, 16, 24), (1000, 1000, 1), (256, 256, 256), (64, 400, 3)]


@pytest.mark.parametrize("tile", sorted(DIMS))
@pytest.mark.parametrize("n", GRIDS, ids=lambda n: "x".join(map(str, n)))
def test_depths_follow_the_blocks(tile, n):
    d = depths(tile, n)
    assert d and d == sorted(set(d)) and all(k <= n[2] for k in d[1:])
    for kz in (6, 8, 12, 16, 32, 64):                       # deep ones wherever they give half the CUs a block
        assert (kz in d) == (kz <= n[2] and 2 * blocks(tile, n, kz) >= NCU), kz
    for kz in (2, 3):                                       # shallow ones where depth 4 leaves CUs short of blocks
        if kz < n[2]:
            assert (kz in d) == (blocks(tile, n, 4) < 4 * NCU), kz
    assert n[2] < 4 or 4 in d


def test_a_narrow_grid_is_offered_deep_marches():
    """1.66e6 voxels of 40 x 40 columns: 64 planes still give the 32 x 8 shape 170 blocks."""
    assert depths(4, (40, 40, 1040)) == [4, 6, 8, 12, 16, 32, 64]


def test_the_device_counts():
    rng = random.Random(2)
    for _ in range(500):
        n, tile = tuple(rng.randint(1, 400) for _ in range(3)), rng.choice(sorted(DIMS))
        assert set(depths(tile, n, 32)) - {2, 3} >= set(depths(tile, n, 256)) - {2, 3}
