"""The denoiser's weight-gradient launch (host arithmetic, CPU only): one round
of the blocks that the device holds at once, each with as many bricks."""
import ctypes as C

import pytest

from tam_amd import lib


@pytest.mark.parametrize("ncu", [32, 128, 256])
@pytest.mark.parametrize("n", [(32, 32, 32), (128, 128, 128), (64, 96, 160), (256, 256, 256)])
@pytest.mark.parametrize("cin,cout,rows", [(16, 16, 1), (48, 16, 3), (16, 32, 3), (32, 32, 6), (96, 32, 18),
                                           (32, 64, 6), (64, 64, 12)])
def test_one_round_of_resident_blocks(ncu, n, cin, cout, rows):
    blocks = lib.load().tam_internal_brick_blocks(ncu, *n, cin, cout)
    bricks = n[2] // 16 * (n[1] // 8) * (n[0] // 4)
    held = ncu * (1 if cout == 64 else 2)
    assert blocks % rows == 0 and blocks <= max(held, rows)
    per = blocks // rows
    each = -(-bricks // per)
    assert per <= bricks and each <= -(-bricks // max(1, held // rows))     # no block has more than its share


def test_host_functions_start_a_cache_line():
    """Where they fall in one sets how fast the weights are drawn."""
    L = lib.load()
    for name in lib.EXPORTED + ("tam_dn_create",):
        assert C.cast(getattr(L, name), C.c_void_p).value % 64 == 0, name
