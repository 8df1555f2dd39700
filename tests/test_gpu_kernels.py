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


# one workgroup up to 4,096 pairs, tiles of 1,024 below 192 * 4,096 pairs, of 4,096 from there
@pytest.mark.parametrize("n", [4095, 4096, 4097, 5120, 5121, 192 * 4096 - 1, 192 * 4096, 193 * 4096 + 1])
@pytest.mark.parametrize("bits", [32, 64])
def test_sort_tile_sizes(ctx, n, bits):
    """Stable order of few distinct keys and of random ones, whole and partial bit ranges."""
    rng = np.random.default_rng(n + bits)
    dt = np.uint64 if bits == 64 else np.uint32
    for keys, end in ((rng.integers(0, 7, n).astype(dt), 3), (rng.integers(0, 1 << (bits - 1), n).astype(dt), bits - 3)):
        d = [ctx.upload(a) for a in (keys, np.arange(n, dtype=np.uint32), np.zeros_like(keys), np.zeros(n, np.uint32))]
        try:
            ctx.sort_pairs(d[0], d[1], d[2], d[3], n, bits, end)
            got = ctx.download(d[3], (n,), np.uint32)
            gk = ctx.download(d[2], (n,), dt)
        finally:
            for p in d:
                ctx.free(p)
        order = np.argsort(keys & dt((1 << end) - 1), kind="stable")
        assert np.array_equal(got, order.astype(np.uint32)) and np.array_equal(gk, keys[order])


def test_exact_rounds_of_all_small_sizes(ctx, oracle):
    """A captured round is replayed for every number of points that shares
    its grids: exact mode, sizes falling and rising, against the oracle."""
    pts = np.random.default_rng(11).random((340, 3)).astype(np.float32)
    cfg = wtet_amd.Config(predicate_mode="exact")
    for n in list(range(330, 20, -9)) + list(range(20, 330, 7)):
        got = oracle.canonical_real(ctx.delaunay(pts[:n], cfg).tets, n)
        want = oracle.canonical_real(oracle.delaunay(oracle.normalize_points(pts[:n])[0]), n)
        assert np.array_equal(got, want), n


# 2,048 points (512 in exact mode) end the one-workgroup rounds; lists of more
# than 1,024 (128) entries leave them within a run, and so do too few slots
@pytest.mark.parametrize("n", [4, 5, 64, 512, 513, 2047, 2048, 2049])
@pytest.mark.parametrize("kw", [{}, {"predicate_mode": "exact"}, {"presize": "grow"},
                                {"enable_hilbert_sorting": True, "collect_stats": True}])
def test_rounds_in_one_workgroup(ctx, oracle, n, kw):
    """The mesh of few points, and the same mesh cut short by the round limit
    and finished by the host, against the oracle."""
    rng = np.random.default_rng(n)
    p = rng.random((n, 3)).astype(np.float32)
    p[n // 2:] = p[n // 2:] * np.float32(0.05) + np.float32(0.4)
    p[-1] = p[0] if n > 64 else p[-1]
    want = oracle.canonical_real(oracle.delaunay(oracle.normalize_points(p)[0]), n)
    for extra in ({}, {"max_insert_iterations": 7}):
        r = ctx.delaunay(p, wtet_amd.Config(**kw, **extra))
        assert np.array_equal(oracle.canonical_real(r.tets, n), want), (n, kw, extra)
        assert r.stats["rounds"] <= extra.get("max_insert_iterations", 100)


def test_batch_of_few_points_in_all(ctx, oracle):
    """Clouds that share the one-workgroup rounds: 40 of 4 to 45 points."""
    rng = np.random.default_rng(3)
    clouds = [rng.random((4 + i, 3)).astype(np.float32) for i in range(40)]
    r = ctx.delaunay_batch(clouds)
    for c, p in zip(range(40), clouds):
        want = oracle.canonical_real(oracle.delaunay(oracle.normalize_points(p)[0]), len(p))
        assert np.array_equal(oracle.canonical_real(r[c].tets, len(p)), want), c


@pytest.mark.parametrize("n", [700, 3000, 20000])
@pytest.mark.parametrize("iters", [1, 2, 5])
@pytest.mark.parametrize("mode", ["filtered", "exact"])
def test_flip_lists_left_over_rounds(ctx, oracle, n, iters, mode):
    """Few flip iterations a round: most of the list waits over the splits of
    the next rounds, and each tet has to stand in it once."""
    p = np.random.default_rng(n + iters).random((n, 3)).astype(np.float32)
    r = ctx.delaunay(p, wtet_amd.Config(max_flip_iterations=iters, predicate_mode=mode))
    want = oracle.canonical_real(oracle.delaunay(oracle.normalize_points(p)[0]), n)
    assert np.array_equal(oracle.canonical_real(r.tets, n), want)


@pytest.mark.parametrize("side,extra", [(12, 0), (13, 0), (20, 0), (20, 12000)])
def test_lattices_that_take_the_full_predicates(ctx, oracle, side, extra):
    """Inputs whose tets the filters leave: below and above the size of the
    one-workgroup rounds, and mixed with points in general position."""
    g = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3).astype(np.float32)
    rng = np.random.default_rng(side + extra)
    p = np.concatenate([g, rng.random((extra, 3)).astype(np.float32) * (side - 1) + np.float32(side)])
    p = p[rng.permutation(len(p))].astype(np.float32)
    want = oracle.canonical_real(oracle.delaunay(oracle.normalize_points(p)[0]), len(p))
    for _ in range(3):  # launched, recorded and replayed
        assert np.array_equal(oracle.canonical_real(ctx.delaunay(p).tets, len(p)), want)


# around a wave, the one-workgroup rounds (2,048 points) and several workgroups
@pytest.mark.parametrize("n", [4, 63, 64, 65, 2048, 2049, 30000])
def test_first_vote_takes_the_deepest_point(ctx, oracle, n):
    """All points lie in one tet: the round's one winner is the point deepest
    inside its circumsphere.  Depths are compared in f32 on the device: two
    roundings of 2^-24 (the f64 error is far below)."""
    p = np.random.default_rng(n).random((n, 3)).astype(np.float32)
    r = ctx.delaunay(p, wtet_amd.Config(max_insert_iterations=1, enable_splaying=False))
    won = np.unique(r.tets[r.tets < n])
    assert len(won) == 1 and r.stats["rounds"] == 1
    V = oracle.extended_points(oracle.normalize_points(p)[0])
    s = V[n:n + 4]
    c = np.linalg.solve(2 * (s[1:] - s[0]), (s[1:] ** 2).sum(1) - (s[0] ** 2).sum())
    depth = ((s[0] - c) ** 2).sum() - ((V[:n] - c) ** 2).sum(1)
    assert depth[won[0]] >= depth.max() * (1 - 2 * 2.0 ** -24)


# counts of 256 points or slots in one scan, four to a load
@pytest.mark.parametrize("n", [255, 1023, 1025, 32769])
def test_block_scan_remainders(ctx, oracle, n):
    p = np.random.default_rng(n).random((n, 3)).astype(np.float32)
    want = oracle.canonical_real(oracle.delaunay(oracle.normalize_points(p)[0]), n)
    assert np.array_equal(oracle.canonical_real(ctx.delaunay(p).tets, n), want)


def test_block_scan_of_several_steps(ctx):
    """1.4M points have over the 32,768 blocks of slots that one step takes:
    every point is a vertex and the adjacency is closed."""
    n = 1400000
    p = np.random.default_rng(9).random((n, 3)).astype(np.float32)
    r = ctx.delaunay(p)
    assert len(np.unique(r.tets[r.tets < n])) == n
    t, f = r.adjacency >> 5, r.adjacency & 3
    inner = r.adjacency != 0xFFFFFFFF
    rows = np.repeat(np.arange(len(t), dtype=np.uint32)[:, None], 4, 1)
    faces = np.tile(np.arange(4, dtype=np.uint32), (len(t), 1))
    back = r.adjacency[t[inner], f[inner]]
    assert np.array_equal(back >> 5, rows[inner]) and np.array_equal(back & 3, faces[inner])


# a histogram block for 8,192 keys, from 256 to 1,024 of them; digits that all
# lanes of a wave share, and that few do
@pytest.mark.parametrize("n", [257 * 8192 - 1, 257 * 8192, 1025 * 8192 + 1])
@pytest.mark.parametrize("distinct", [1, 3, 4096])
def test_sort_histogram_blocks_and_ties(ctx, n, distinct):
    keys = np.random.default_rng(n + distinct).integers(0, distinct, n).astype(np.uint32) + np.uint32(7)
    d = [ctx.upload(a) for a in (keys, np.arange(n, dtype=np.uint32), np.zeros_like(keys), np.zeros(n, np.uint32))]
    try:
        ctx.sort_pairs(d[0], d[1], d[2], d[3], n, 32, 13)
        got = ctx.download(d[3], (n,), np.uint32)
    finally:
        for p in d:
            ctx.free(p)
    assert np.array_equal(got, np.argsort(keys, kind="stable").astype(np.uint32))
