"""Which kernels a triangulation takes, by the launches the context counts."""
import numpy as np
import pytest

import wtet_amd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = wtet_amd.Context(0)
    yield c
    c.close()


def _lattice(side):
    g = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)
    return (g / max(side - 1, 1)).astype(np.float32)


def _launches(ctx, run):
    ctx.set_profiling(True)
    try:
        r = run()
        return r, {k: v[0] for k, v in ctx.kernel_times().items()}
    finally:
        ctx.set_profiling(False)


@pytest.mark.parametrize("side", [8, 9])
def test_crowded_rounds_leave_the_workgroup(ctx, oracle, side):
    """Rounds that leave hundreds of entries an iteration to the full
    predicates go to the list kernels until they fit one workgroup again: the
    one-workgroup kernels run before and after them, not once more for each
    such round (three launches and more)."""
    runs = []
    for seed in range(4):
        p = _lattice(side)[np.random.default_rng(seed).permutation(side ** 3)]
        r, n = _launches(ctx, lambda: ctx.delaunay(p))
        runs.append(n)
        want = oracle.canonical_real(oracle.delaunay(oracle.normalize_points(p)[0]), len(p))
        assert np.array_equal(oracle.canonical_real(r.tets, len(p)), want)
    # a round's list may fall below the bound and rise over it again: half a launch more on average
    assert sum(n["flip_small"] for n in runs) <= 2.5 * len(runs), runs
    assert all(n["flip_check"] for n in runs), runs
