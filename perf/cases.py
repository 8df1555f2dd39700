"""The work that programs give this library, as cases that can be timed.

A case is a dict of plain values.  ``prepare`` makes what a program holds
before the call (points of a seed, the device context), ``run`` is one pass
through the public entry points.

The rows of a triangulation come in an order that differs from run to run
(the device fills lists with atomics), so a program that stores, compares or
indexes meshes puts them in canonical order first: vertices ascending within a
tet, tets ascending; where it wants the neighbours too, the vertex across
each face in the same order.
``run`` returns the whole mesh in that form, in buffers sized for the number
of points alone (rows past the mesh hold -1), as a program with static shapes
keeps them.
"""
import math

import numpy as np
import torch

import wtet_amd
from wtet_amd import presize

_ctx = None


def context():
    """One device context per process, as a serving program keeps it."""
    global _ctx
    if _ctx is None:
        _ctx = wtet_amd.Context(0)
    return _ctx


def listed():
    return [
        # one small neighbourhood at a time: latency of a call, host points
        # in, host mesh out
        {"name": "tiny_64_host", "kind": "cloud", "api": "host", "dist": "uniform", "n": 64},
        # an object scan cut into parts, ragged size
        {"name": "clusters_1k_host", "kind": "cloud", "api": "host", "dist": "clusters", "n": 1003},
        # the 10,000-point benchmark configuration: Hilbert order, exact only
        {"name": "hilbert_exact_10k", "kind": "cloud", "api": "resident", "dist": "uniform", "n": 10000,
         "exact": True, "hilbert": True},
        # an ordinary cloud, host points in, host mesh out (PCIe both ways)
        {"name": "uniform_100k_host", "kind": "cloud", "api": "host", "dist": "uniform", "n": 100000},
        # the headline benchmark: 1M uniform points resident on the device
        {"name": "uniform_1M", "kind": "cloud", "api": "resident", "dist": "uniform", "n": 1000000},
        # anisotropic densities, slots sized by the presizing network
        {"name": "anisotropic_2M_learned", "kind": "cloud", "api": "resident", "dist": "anisotropic",
         "n": 1999993, "learned": True},
        # surface samples: near-cospherical, many faces the flips leave stuck
        {"name": "sphere_50k", "kind": "cloud", "api": "resident", "dist": "sphere", "n": 50021},
        # degenerate stress: the points of a grid in a random order
        {"name": "lattice_48", "kind": "cloud", "api": "resident", "dist": "lattice", "n": 48 ** 3},
        # a batch of many clouds from host memory
        {"name": "batch_64_host", "kind": "batch", "api": "host", "clouds": 64, "median": 2000.0},
        # the batched configuration (log-normal sizes around 2,000 points)
        {"name": "batch_2048", "kind": "batch", "api": "resident", "clouds": 2048, "median": 2000.0},
        # presizing network: loss and gradient of one large minibatch
        {"name": "presize_grad_2048", "kind": "grad", "rows": 2048},
        # the library's stable sort on 63-bit point keys
        {"name": "sort_4M", "kind": "sort", "n": 4000037, "key_bits": 64, "end_bit": 63},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    x = rng.random()
    if x < 0.70:
        dist = rng.choice(["uniform", "uniform", "clusters", "anisotropic", "sphere", "lattice"])
        c = {"kind": "cloud", "api": rng.choice(["host", "resident"]), "dist": dist}
        if dist == "lattice":
            c["n"] = rng.randint(4, 48) ** 3
        else:
            c["n"] = _log_uniform(rng, 16, {"sphere": 50000}.get(dist, 1500000))
        if rng.random() < 0.2:
            c["hilbert"] = True
        if c["n"] <= 20000 and rng.random() < 0.25:
            c["exact"] = True
        if dist != "lattice" and rng.random() < 0.2:
            c["learned"] = True
        return c
    if x < 0.86:
        return {"kind": "batch", "api": rng.choice(["host", "resident"]), "clouds": _log_uniform(rng, 2, 1500),
                "median": float(_log_uniform(rng, 100, 2000))}
    if x < 0.93:
        return {"kind": "grad", "rows": rng.randint(64, 4096)}
    bits = rng.choice([32, 64])
    return {"kind": "sort", "n": _log_uniform(rng, 1000, 4000000), "key_bits": bits,
            "end_bit": rng.randint(8, bits)}


# -- inputs ------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _points(dist, n, seed):
    """(n, 3) f32 device points: the benchmark's distributions."""
    g = _gen(seed)
    rand = lambda *s: torch.rand(*s, generator=g, device="cuda")  # noqa: E731
    randn = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    if dist == "uniform":
        return rand(n, 3)
    if dist == "sphere":
        p = randn(n, 3).double()
        return (p / p.norm(dim=1, keepdim=True)).float().contiguous()
    if dist == "lattice":
        k = int(round(n ** (1 / 3)))
        i = torch.arange(k, device="cuda", dtype=torch.float32) / max(k - 1, 1)
        p = torch.cartesian_prod(i, i, i)
        return p[torch.randperm(n, generator=g, device="cuda")].contiguous()
    if dist == "clusters":  # isotropic Gaussians, samples outside the box redrawn
        k = 1 + seed % 8
        centers, sig = rand(k, 3), 0.02 + 0.18 * rand(k)
        parts, have = [], 0
        while have < n:
            c = torch.randint(0, k, (2 * n,), generator=g, device="cuda")
            s = centers[c] + randn(2 * n, 3) * sig[c, None]
            s = s[((s >= 0) & (s <= 1)).all(1)]
            parts.append(s)
            have += len(s)
        return torch.cat(parts)[:n].contiguous()
    # anisotropic: 32 rotated Gaussians and a tenth of uniform points
    k, nu = 32, n // 10
    m = n - nu
    centers, q = rand(k, 3), torch.linalg.qr(randn(k, 3, 3))[0]
    scale = (1e-4 + (1e-2 - 1e-4) * rand(k, 3)).sqrt()
    parts, have = [], 0
    while have < m:
        c = torch.randint(0, k, (2 * m,), generator=g, device="cuda")
        z = randn(2 * m, 3) * scale[c]
        s = centers[c] + (q[c] * z[:, None, :]).sum(2)
        s = s[((s >= 0) & (s <= 1)).all(1)]
        parts.append(s)
        have += len(s)
    p = torch.cat([torch.cat(parts)[:m], rand(nu, 3)])
    return p[torch.randperm(n, generator=g, device="cuda")].contiguous()


def _batch_sizes(case):
    """Log-normal cloud sizes (sigma 0.63, in 64..50000), the same for every seed."""
    rng = np.random.default_rng(1234)
    z = rng.normal(math.log(case["median"]), 0.63, case["clouds"])
    return np.clip(np.rint(np.exp(z)), 64, 50000).astype(np.int64)


def _batch_points(sizes, seed):
    """Each cloud a mixture of up to 8 Gaussians folded back into the unit box."""
    g = _gen(seed)
    C, n = len(sizes), int(sizes.sum())
    k = torch.randint(1, 9, (C,), generator=g, device="cuda")
    centers = torch.rand(C, 8, 3, generator=g, device="cuda")
    sig = 0.02 + 0.18 * torch.rand(C, 8, generator=g, device="cuda")
    c = torch.repeat_interleave(torch.arange(C, device="cuda"), torch.from_numpy(sizes).cuda())
    j = (torch.rand(n, generator=g, device="cuda") * k[c]).long().clamp_(max=7)
    p = centers[c, j] + torch.randn(n, 3, generator=g, device="cuda") * sig[c, j, None]
    p = p.abs() % 2.0
    return torch.where(p > 1, 2 - p, p).contiguous()


def prepare(case, seed):
    ctx = context()
    if case["kind"] == "cloud":
        cfg = wtet_amd.Config(predicate_mode="exact" if case.get("exact") else "filtered",
                              enable_hilbert_sorting=bool(case.get("hilbert")),
                              presize="learned" if case.get("learned") else "fixed")
        p = _points(case["dist"], case["n"], seed)
        if case["api"] == "host":
            p = p.cpu().numpy()
        return {"case": case, "ctx": ctx, "cfg": cfg, "points": p}
    if case["kind"] == "batch":
        sizes = _batch_sizes(case)
        off = np.zeros(len(sizes) + 1, np.uint64)
        off[1:] = np.cumsum(sizes)
        p = _batch_points(sizes, seed)
        if case["api"] == "host":
            p = p.cpu().numpy()
        return {"case": case, "ctx": ctx, "cfg": wtet_amd.Config(), "points": p, "offsets": off}
    if case["kind"] == "grad":
        # features as the library makes them (sparse occupancy histograms,
        # moments, log n), targets around the shipped network's own scale
        params = presize.load_model()
        rng = np.random.default_rng(seed)
        rows, F = case["rows"], wtet_amd._core.PRESIZE_FEATURES
        h = rng.gamma(0.2, 1.0, (rows, 512))
        feat = np.empty((rows, F), np.float32)
        feat[:, :512] = h / h.sum(1, keepdims=True)
        feat[:, 512:515] = rng.uniform(0.3, 0.7, (rows, 3))
        feat[:, 515:518] = rng.uniform(0.01, 0.1, (rows, 3))
        feat[:, 518:521] = rng.uniform(-0.02, 0.02, (rows, 3))
        feat[:, 521] = rng.uniform(math.log(100), math.log(2e6), rows)
        tgt = np.stack([rng.normal(1.9, 0.2, rows), rng.normal(0.5, 0.4, rows),
                        np.abs(rng.normal(3.0, 2.0, rows))], 1).astype(np.float32)
        return {"case": case, "ctx": ctx, "params": params, "feat": feat, "tgt": tgt}
    g = _gen(seed)
    n, bits, end = case["n"], case["key_bits"], case["end_bit"]
    dt = torch.int64 if bits == 64 else torch.int32
    raw = torch.randint(0, 1 << min(end, 62), (n,), generator=g, device="cuda", dtype=torch.int64)
    if end > 62:  # the bits above the generator's range
        raw = (raw << (end - 62)) | torch.randint(0, 1 << (end - 62), (n,), generator=g, device="cuda")
    keys = raw.to(dt)
    return {"case": case, "ctx": ctx, "keys": keys, "vals": torch.arange(n, device="cuda", dtype=torch.int32),
            "keys_out": torch.empty_like(keys), "vals_out": torch.empty(n, device="cuda", dtype=torch.int32)}


# -- passes ------------------------------------------------------------------------

def _ascending(tets):
    """The four columns of the rows, each row ascending."""
    a, b, c, d = tets.unbind(1)
    a, b = torch.minimum(a, b), torch.maximum(a, b)
    c, d = torch.minimum(c, d), torch.maximum(c, d)
    a, c = torch.minimum(a, c), torch.maximum(a, c)
    b, d = torch.minimum(b, d), torch.maximum(b, d)
    b, c = torch.minimum(b, c), torch.maximum(b, c)
    return a, b, c, d


def _sorted_keys(a, b, c, bits, cloud=None, void=None):
    """Sorted keys of the rows' three smallest vertices (and their cloud), and
    the order; rows marked void go last."""
    key = ((a.long() << bits | b) << bits) | c
    if cloud is not None:
        key |= cloud << 3 * bits
    if void is not None:
        key.masked_fill_(void, torch.iinfo(torch.int64).max)
    return torch.sort(key)


def _swaps(key, d):
    """Where rows i and i + 1 share their three smallest vertices (two rows do
    at most) and must change places for the fourth to ascend."""
    return (key[1:] == key[:-1]) & (d[:-1] > d[1:])


def _padded(x, rows):
    p = torch.full((rows,) + x.shape[1:], -1, dtype=x.dtype, device="cuda")
    p[:len(x)] = x
    return p


def _packed(tets, bits, rows, count, cloud=None, void=None):
    """The mesh's tets as (cloud, three smallest vertices) in one word and the
    fourth vertex in another."""
    a, b, c, d = _ascending(tets)
    key, perm = _sorted_keys(a, b, c, bits, cloud, void)
    key, d = key[:count], d[perm[:count]]
    swap = _swaps(key, d)
    e = d.clone()
    e[:-1] = torch.where(swap, d[1:], d[:-1])
    e[1:] = torch.where(swap, d[:-1], e[1:])
    return {"abc": _padded(key, rows), "d": _padded(e, rows), "num_tets": count}


def _with_neighbours(tets, adj, bits, rows):
    """Sorted vertices and, across the face opposite each of them, the
    neighbour's vertex."""
    across = tets.view(-1)[((adj >> 5).long() << 2) + (adj & 3)]
    a, b, c, d = _ascending(tets << 2 | torch.arange(4, device="cuda", dtype=torch.int32))
    key, perm = _sorted_keys(a >> 2, b >> 2, c >> 2, bits)
    swap = _swaps(key, d[perm])
    at = torch.arange(len(perm), device="cuda")
    at[:-1] += swap
    at[1:] -= swap.long()
    perm = perm[at]
    s = torch.stack([a, b, c, d], 1)[perm]
    return {"tets": _padded(s >> 2, rows), "across": _padded(across[perm].gather(1, (s & 3).long()), rows),
            "num_tets": len(perm)}


def run(state):
    case, ctx = state["case"], state["ctx"]
    if case["kind"] == "cloud":
        n = case["n"]
        bits, rows = (n + 4).bit_length(), 8 * n + 64  # general position has about 6.8 n
        if case["api"] == "host":
            r = wtet_amd.delaunay(state["points"], state["cfg"])
            tets = torch.from_numpy(r.tets.view(np.int32)).cuda()
            adj = torch.from_numpy(r.adjacency.view(np.int32)).cuda()
            return _with_neighbours(tets, adj, bits, rows)
        torch.cuda.current_stream().synchronize()  # the points are this stream's
        m, dt, _ = ctx.delaunay_resident(state["points"].data_ptr(), n, state["cfg"])
        tets = torch.empty((m, 4), dtype=torch.int32, device="cuda")
        ctx.copy(tets.data_ptr(), dt, m * 16)  # the context reuses its rows
        return _packed(tets, bits, rows, m)
    if case["kind"] == "batch":
        off = state["offsets"]
        C, n = len(off) - 1, int(off[-1])
        bits, rows = (int(np.diff(off.astype(np.int64)).max()) + 4).bit_length(), 8 * n + 64 * C
        if case["api"] == "host":
            r = ctx.delaunay_batch(state["points"], off, state["cfg"])
            tets = torch.from_numpy(r.tets.view(np.int32)).cuda()
            start, count = r.tet_offsets[:-1].astype(np.int64), np.diff(r.tet_offsets.astype(np.int64))
        else:
            torch.cuda.current_stream().synchronize()
            dt, _, start, count = ctx.delaunay_batch_resident(state["points"].data_ptr(), off, state["cfg"])
            start, count = start.astype(np.int64), count.astype(np.int64)
            m = int((start + count).max())
            tets = torch.empty((m, 4), dtype=torch.int32, device="cuda")
            ctx.copy(tets.data_ptr(), dt, m * 16)
        # the cloud of each row; rows before, between and after the clouds' own
        # (a repaired cloud's rows come after the others, its old ones stay)
        # are void
        order = np.argsort(start, kind="stable")
        begin = start[order]
        begin[0] = 0  # the first cloud's old rows, when it was repaired
        span = np.diff(np.append(begin, len(tets)))
        gaps = int(span.sum() - count.sum())
        order, span = torch.from_numpy(order).cuda(), torch.from_numpy(span).cuda()
        cloud = torch.repeat_interleave(order, span, output_size=len(tets))
        void = None
        if gaps:
            row = torch.arange(len(tets), device="cuda")
            first, end = torch.from_numpy(start).cuda(), torch.from_numpy(start + count).cuda()
            void = (row < first[cloud]) | (row >= end[cloud])
        mesh = _packed(tets, bits, rows, int(count.sum()), cloud, void)
        mesh["tets_per_cloud"] = torch.from_numpy(count)
        return mesh
    if case["kind"] == "grad":
        loss, grad = ctx.mlp_loss_grad(state["params"], state["feat"], state["tgt"])
        return {"loss": np.float32(loss), "grad": grad}
    torch.cuda.current_stream().synchronize()
    ctx.sort_pairs(state["keys"].data_ptr(), state["vals"].data_ptr(), state["keys_out"].data_ptr(),
                   state["vals_out"].data_ptr(), case["n"], case["key_bits"], case["end_bit"])
    return state["keys_out"], state["vals_out"]


def exact(case, seed):
    """The gradient case in 64 bits; the other outputs are whole numbers."""
    if case["kind"] != "grad":
        return None
    s = prepare(case, seed)
    p = s["params"].astype(np.float64)
    w = {k: p[a:b] for k, (a, b) in presize.OFF.items()}
    W1, W2, W3 = w["W1"].reshape(-1, 128), w["W2"].reshape(128, 128), w["W3"].reshape(128, 3)
    x = (s["feat"].astype(np.float64) - w["fmean"]) / w["fstd"]
    y = (s["tgt"].astype(np.float64) - w["tmean"]) / w["tstd"]
    z1 = x @ W1 + w["b1"]
    h1 = np.maximum(z1, 0)
    z2 = h1 @ W2 + w["b2"]
    h2 = np.maximum(z2, 0)
    e = h2 @ W3 + w["b3"] - y
    g = np.zeros_like(p)

    def put(name, v):
        a, b = presize.OFF[name]
        g[a:b] = np.ravel(v)

    d3 = 2 * e / e.size
    d2 = (d3 @ W3.T) * (z2 > 0)
    d1 = (d2 @ W2.T) * (z1 > 0)
    put("W3", h2.T @ d3)
    put("b3", d3.sum(0))
    put("W2", h1.T @ d2)
    put("b2", d2.sum(0))
    put("W1", x.T @ d1)
    put("b1", d1.sum(0))
    return {"loss": np.float64(np.mean(e * e)), "grad": g}


def work(case):
    """Input read once, result written once; a mesh of n points in general
    position has about 6.77 n tets of 32 bytes (vertices and adjacency), and
    each point and tet is visited at least once by an insphere test (about
    100 operations)."""
    if case["kind"] == "cloud":
        rows = 6.77 * case["n"]
        return {"bytes": 12.0 * case["n"] + 32.0 * rows, "flops": 4 * 100.0 * rows / 2}
    if case["kind"] == "batch":
        n = float(_batch_sizes(case).sum())
        return {"bytes": 12.0 * n + 32.0 * 6.77 * n, "flops": 4 * 100.0 * 6.77 * n / 2}
    if case["kind"] == "grad":
        r = float(case["rows"])
        macs = r * (522 * 128 + 128 * 128 + 128 * 3)
        return {"bytes": 4.0 * (r * 525 + 2 * 84896), "flops": 2 * macs * 3 - 2 * r * 522 * 128}
    pair = case["key_bits"] // 8 + 4
    return {"bytes": 2.0 * case["n"] * pair, "flops": 0.0}
