"""Kernels at the sizes where their tiling can go wrong."""
import numpy as np
import pytest

import wtet_amd
from oracle import mlp_ref as R
from wtet_amd import presize

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = wtet_amd.Context(0)
    yield c
    c.close()


# row tiles of 16, gradient slices of 256, the largest batch
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 64, 255, 256, 257, 1000, 4096])
def test_gradient_row_tiles_and_slices(ctx, rows):
    """Loss and gradient against the FP64 reference.  Every sum has at most
    about 200 FP32 roundings in a chain (64 rows per wave, 4 waves, 16
    slices; 522 features in steps of 4), 200 * 2^-24 = 1.2e-5 of the summed
    magnitudes, which stay within a few times the largest entry: 1e-4."""
    rng = np.random.default_rng(rows)
    X = np.empty((rows, wtet_amd._core.PRESIZE_FEATURES), np.float32)
    X[:, :512] = rng.random((rows, 512)) / 256
    X[:, 512:] = rng.uniform(0.1, 0.9, (rows, 10))
    Y = rng.normal(0.0, 1.0, (rows, 3)).astype(np.float32)
    stat = np.random.default_rng(7)
    p = presize.init_params(stat.random((64, X.shape[1])), stat.normal(size=(64, 3)), 3)
    a, b = presize.OFF["b1"]
    p[a:b] = stat.normal(0.0, 0.5, b - a)
    loss, g = ctx.mlp_loss_grad(p, X, Y)
    lref, gref = R.loss_grad(p.astype(np.float64), X.astype(np.float64), Y.astype(np.float64))
    assert loss == pytest.approx(lref, rel=1e-4)
    scale = np.abs(gref).max()
    assert np.abs(g - gref).max() <= 1e-4 * scale, np.abs(g - gref).max() / scale
