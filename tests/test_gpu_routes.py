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


def test_lattices_in_a_batch_do_not_settle_the_other_clouds_route(ctx, oracle):
    """Small lattices leave most of the first rounds' tets to the full
    predicates; once they are done, a cloud of points in general position goes
    back to the filters, whose deferred check is then launched in every round
    (in the first one alone when the early rounds settled the route)."""
    rng = np.random.default_rng(5)
    clouds = [_lattice(8)[rng.permutation(512)] for _ in range(64)] + [rng.random((30000, 3)).astype(np.float32)]
    r, n = _launches(ctx, lambda: ctx.delaunay_batch(clouds))
    for c in (0, 63, 64):
        p = clouds[c]
        want = oracle.canonical_real(oracle.delaunay(oracle.normalize_points(p)[0]), len(p))
        assert np.array_equal(oracle.canonical_real(r[c].tets, len(p)), want), c
    assert n["flip_check_deferred"] >= r.stats["rounds"] // 3, n
