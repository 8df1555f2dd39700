"""Device workspaces that one call shares between stages of different sizes,
on contexts that no larger call has grown before."""
import ctypes
import time

import numpy as np
import pytest

import wtet_amd

pytestmark = pytest.mark.gpu


# 800,000 points are sorted in tiles of 4,096, the 780,000 left without the
# duplicates (reordered in the same workspace) in tiles of 1,024
@pytest.mark.parametrize("batch", [False, True])
def test_hilbert_order_of_fewer_points_than_were_sorted(batch):
    n, dup = 800000, 20000
    rng = np.random.default_rng(21)
    p = rng.random((n, 3)).astype(np.float32)
    p[n - dup:] = p[:dup]
    cfg = wtet_amd.Config(enable_hilbert_sorting=True)
    cut = n - 1000  # the second cloud of the batch; no duplicates within it
    print("hilbert n=%d duplicates=%d batch=%s" % (n, dup, batch), flush=True)
    ctx = wtet_amd.Context(0)
    try:
        if batch:
            res = ctx.delaunay_batch([p[:cut], p[cut:]], config=cfg)
            clouds = [(p[:cut], res[0]), (p[cut:], res[1])]
        else:
            clouds = [(p, ctx.delaunay(p, cfg))]
    finally:
        ctx.close()
    for q, r in clouds:
        used = np.unique(r.tets[r.tets < len(q)])
        assert len(used) == len(np.unique(q, axis=0))
        bad, interior = wtet_amd.check_quality(q, r)
        assert bad == 0 and interior > 6 * len(used)


def _free_bytes():
    """Free device memory, from the HIP runtime that the library loaded."""
    hip = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL(hip).hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_training_gives_a_large_set_back():
    """The features of 100,000 rows (209 MB) are not kept once the training is
    over; what is, is at most 64 MiB."""
    from wtet_amd import presize
    rows, batch = 100000, 1024
    rng = np.random.default_rng(2)
    X = rng.random((rows, wtet_amd._core.PRESIZE_FEATURES), dtype=np.float32)
    Y = rng.random((rows, 3), dtype=np.float32)
    ctx = wtet_amd.Context(0)
    try:
        p = presize.init_params(X[:4096], Y[:4096], 3)
        small, _ = ctx.mlp_train(p, X[:2048], Y[:2048], epochs=1, batch=batch, lr=1e-3)
        before = _free_bytes()
        big, _ = ctx.mlp_train(p, X, Y, epochs=1, batch=batch, lr=1e-3)
        for _ in range(50):  # the driver reports freed memory a moment later
            if before - _free_bytes() <= 64 << 20:
                break
            time.sleep(0.1)
        assert before - _free_bytes() <= 64 << 20
        again, _ = ctx.mlp_train(p, X[:2048], Y[:2048], epochs=1, batch=batch, lr=1e-3)
    finally:
        ctx.close()
    assert np.all(np.isfinite(big)) and np.array_equal(small, again)
