"""Which field downloads take the pinned ring (host arithmetic, CPU only): a
ring pays for results of 2 MiB and more; below, a plain copy is faster but for
the smallest fields, which take a ring only where one is idle."""
import pytest

from tam_amd import lib

F64, F32, U8 = range(3)
PLAIN, IDLE, RING = range(3)
KIB = 1024 // 8                                            # doubles


@pytest.mark.parametrize("kind,kib,route", [(F64, 4, IDLE), (F64, 32, PLAIN), (F64, 256, PLAIN), (F64, 1447, PLAIN),
                                            (F64, 2048, RING), (F64, 65536, RING), (F32, 4, IDLE), (F32, 140, IDLE),
                                            (F32, 256, PLAIN), (F32, 2048, RING), (U8, 108, IDLE), (U8, 172, PLAIN),
                                            (U8, 2048, RING)])
def test_route(kind, kib, route):
    f = lib.load().tam_internal_stage_route
    assert f(kind, lib.C.c_int64(kib * KIB)) == route


@pytest.mark.parametrize("kind,low", [(F64, 16), (F32, 160), (U8, 160)])
def test_lines(kind, low):
    f = lib.load().tam_internal_stage_route
    assert [f(kind, lib.C.c_int64(n)) for n in (1, low * KIB - 1, low * KIB, 2048 * KIB - 1, 2048 * KIB)] == \
        [IDLE, IDLE, PLAIN, PLAIN, RING]
