"""The transport kernel's two ways of finding mu_t -- from the material table
in LDS, or from the per-voxel array (any upload of rhokap selects it) -- and
its split of short runs over waves: the same packets, so the same integer
fates, and tallies that differ by the order of FP64 adds alone (1e-9)."""
import numpy as np
import pytest

from tam_amd import configs, lib

pytestmark = pytest.mark.gpu

SHAPES = {"odd": (37, 51, 45), "one-plane": (64, 40, 1), "row": (33, 1, 7)}


def _problem(n, nmat, crater):
    prob = configs.three_layer_skin(n=n, ext=(0.5, 0.5, 0.25), packets=1, steps=1)
    if nmat > 3:                                     # more materials than the table in LDS holds
        prob.table = [(2.0 + 0.1 * m, 150.0 + m, 0.8, 1.4) for m in range(nmat)]
        prob.mat = (np.arange(prob.mat.size) % nmat).astype(np.uint8).reshape(prob.mat.shape)
    g = prob.grid()
    if crater:
        nz, ny, nx = prob.mat.shape
        hot = np.array(prob.temp)
        hot[1 + nz // 2:nz + 1, 1 + ny // 3:1 + ny // 2, 1 + nx // 3:1 + nx // 2] = prob.params.ablate_K + 5.0
        g.upload(lib.FIELD_TEMP, hot)
        g.rebuild()
    return g


def _fates(s):
    return [s.absorbed, s.specular, s.missed, s.killed, s.crossings, s.interactions, s.tally_adds, s.box_adds] + \
        list(s.escaped)


# packets: one lane, a wave and its neighbours, the 4-a-wave and 64-a-wave
# splits (8 waves a CU on 256 CUs), and both sides of the box's threshold
@pytest.mark.parametrize("packets", [1, 63, 65, 8191, 8193, 131_073, 400_000])
@pytest.mark.parametrize("shape,nmat,crater", [("odd", 3, True), ("odd", 40, False), ("one-plane", 3, False),
                                               ("row", 3, False)])
def test_table_and_array_paths_agree(packets, shape, nmat, crater):
    a, b = (_problem(SHAPES[shape], nmat, crater) for _ in range(2))
    b.upload(lib.FIELD_RHOKAP, b.download(lib.FIELD_RHOKAP))
    for launch, box, fp64 in ((8, True, False), (4, True, True), (3, True, False), (6, True, False), (2, False, False)):
        print("case", packets, shape, nmat, launch, box, fp64, flush=True)
        for g in (a, b):
            g.set_mc_launch(launch, 32)
            g.set_mc_box(box, fp64=fp64)
        sa, sb = (g.mc_run(packets, seed=5, stream=3) for g in (a, b))
        assert _fates(sa) == _fates(sb)
        assert sa.absorbed + sa.specular + sa.missed + sa.killed + sum(sa.escaped) == packets
        ta, tb = (g.download(lib.FIELD_TALLY) for g in (a, b))
        np.testing.assert_allclose(ta, tb, rtol=1e-9, atol=1e-9 * tb.max())
    a.close()
    b.close()
