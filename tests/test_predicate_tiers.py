"""Signs of the exact predicate stages at the edges of their ranges."""
import numpy as np
import pytest

import wtet_amd
from wtet_amd import _core

SUPER = np.array([[-100, -100, -100], [400, -100, -100], [-100, 400, -100], [-100, -100, 400]], np.float32)


def _sets(span, n=400):
    """Sets of five points, mostly coplanar or cospherical, whose differences
    span `span` bits (0: lattice points with one or two super vertices)."""
    rng = np.random.default_rng(span)
    q = rng.integers(0, 3, (n, 5, 3)).astype(np.float32)
    if span:
        far = rng.random((n, 5, 3)) < 0.12
        q = np.where(far, np.float32(2.0 ** (span - 1)), q).astype(np.float32) * np.float32(2.0**-45)
    else:
        q /= np.float32(47)
        for i in range(n):
            two = rng.permutation(5)[: 1 + i % 2]
            q[i, two] = SUPER[rng.permutation(4)[: len(two)]]
    idx = np.stack([rng.permutation(9)[:5] for _ in range(n)]).astype(np.uint32)
    return q, idx


def _check(oracle, run, span, mode):
    q, idx = _sets(span)
    p4, i4 = np.ascontiguousarray(q[:, :4]), np.ascontiguousarray(idx[:, :4])
    d, d4 = q.astype(np.float64), p4.astype(np.float64)
    assert np.array_equal(run(0, p4, i4, mode), oracle.orient3d_sos(d4, i4))
    assert np.array_equal(run(1, q, idx, mode), oracle.orient4d(d, idx))
    assert np.array_equal(run(2, p4, None, mode), oracle.orient3d_sign(d4))
    assert np.array_equal(run(3, q, None, mode), oracle.insphere_sign(d))


# 30 and 41 bits end the two tiers on native integers; 60 the 64-bit limbs
SPANS = [0, 2, 29, 30, 31, 40, 41, 42, 54, 60, 61, 80]


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("span", SPANS)
def test_host_signs_at_tier_edges(oracle, span, mode):
    _check(oracle, _core.predicates_host, span, mode)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("span", SPANS)
def test_device_signs_at_tier_edges(oracle, span, mode):
    c = wtet_amd.Context(0)
    try:
        _check(oracle, lambda *a: c.predicates(*a)[0], span, mode)
    finally:
        c.close()
