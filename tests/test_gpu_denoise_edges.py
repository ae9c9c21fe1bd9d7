"""The denoiser's convolutions at the edges of their staged bricks.

Grids whose three edges differ, so that each side of a brick (16 x 8 x 4
voxels with a ring of one, loaded as two rows at a time and the columns beside
them) falls on a face of the grid in some block, at every level and with the
concatenated inputs.  References and tolerances are those of the kernels'
other tests: 0.6 % of the prediction's range at the worst voxel, 5e-4 at the
median; gradients with cosine similarity >= 0.9999 and a relative L2 error of
at most 6e-3.
"""
import numpy as np
import pytest

import denoise_ref as R
from tam_amd.denoise import Denoiser, param_layout

pytestmark = pytest.mark.gpu


def _inputs(shape, seed):
    rng = np.random.default_rng(seed)
    nz, ny, nx = shape
    base = np.log1p(30.0 * np.exp(-(nz - 1 - np.arange(nz)[:, None, None]) / 6.0)) * np.ones(shape)
    # the faces of the grid stand out: a voxel taken from across one would show
    base[0], base[-1], base[:, 0], base[:, -1], base[:, :, 0], base[:, :, -1] = 2.0, 0.5, 1.5, 3.0, 0.2, 2.5
    f = np.stack([np.maximum(base + 0.3 * rng.standard_normal(shape), 0.0), rng.uniform(-1, 1, shape),
                  rng.uniform(-0.3, 0.5, shape), rng.uniform(-0.5, 0.75, shape)])
    return f.astype(np.float32), base.astype(np.float32)


@pytest.mark.parametrize("shape", [(32, 96, 64), (96, 32, 64), (64, 32, 96)])
def test_forward_and_gradients(shape):
    print("case:", shape, flush=True)
    dn = Denoiser(shape, capacity=1, seed=1)
    p = R.random_params(dn.n, seed=7)
    dn.set_params(p)
    f, target = _inputs(shape, 8)
    out = dn.forward(f)
    ref = R.forward(R.unpack(p), f).detach().numpy()
    span = ref.max() - ref.min()
    err = np.abs(out - ref)
    print("range", span, "max err", err.max(), "median", np.median(err), flush=True)
    assert err.max() <= 6e-3 * span
    assert np.median(err) <= 5e-4 * span
    grads, loss = dn.gradients(f, target)
    dn.close()
    ref_grads, ref_loss = R.gradients(p, f, target)
    assert abs(loss - ref_loss) <= 1e-4 * abs(ref_loss)
    for name, off, shp in param_layout():
        size = int(np.prod(shp))
        a, b = grads[off:off + size].astype(np.float64), ref_grads[off:off + size].astype(np.float64)
        if name == "w0":                      # padding input channels carry no gradient
            a, b = a.reshape(shp)[:, :4].ravel(), b.reshape(shp)[:, :4].ravel()
        nb = np.linalg.norm(b)
        cos = float(a @ b / (np.linalg.norm(a) * nb + 1e-30))
        rel = float(np.linalg.norm(a - b) / (nb + 1e-30))
        print(name, "cos", cos, "rel", rel, flush=True)
        assert cos >= 0.9999 and rel <= 6e-3, name
