"""Device workspaces that one call shares between stages of different sizes,
on contexts that no larger call has grown before."""
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
