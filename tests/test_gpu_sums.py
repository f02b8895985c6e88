"""Rounding of the sums over sources in FP64 where sources run one by one.

The dependencies of every source come from the probe of a tile, which runs the
same kernel, and their sum is exact in math.fsum; what a run is off by is the
rounding of its own additions.  An addition errs by 0.29 ulp (uniform in half an
ulp either way), one that has reached a part p of the sum by p times that.  The
sums in tiles of 64, added up in pairs, and of 300 sources in 5 such tiles, have
(0.2^2 + .. + 1) + 5 0.2^2 (1 + 1/2 + 1/4 + ..) = 2.6 of its squares: 0.47 ulp.
The bound is 1.25 times that."""
import math

import numpy as np
import pytest

import bcx
from test_zz_no_alloc import noalloc

pytestmark = pytest.mark.gpu

BOUND = 1.25 * math.sqrt(2.6 / 12)


def component(n, seed):
    rng = np.random.default_rng(seed)
    e = {(min(i, (i + 1) % n), max(i, (i + 1) % n)) for i in range(n)}
    while len(e) < 3 * n:
        a, b = sorted(map(int, rng.integers(0, n, 2)))
        if a != b:
            e.add((a, b))
    return bcx.Host.from_edges(n, sorted(e)).decompose().components()[0]


def exact(engine, c):
    rows = [engine.debug_tile(c, np.arange(s, min(s + 64, c.n)), precision=bcx.PREC_FP64)[3]
            for s in range(0, c.n, 64)]
    delta = np.concatenate(rows)
    assert delta.shape == (c.n, c.n) and not np.any(c.reach)
    return np.array([math.fsum(delta[:, v]) for v in range(c.n)])


@pytest.mark.parametrize("path", [bcx.PATH_PLAIN, bcx.PATH_BATCHED])
@pytest.mark.parametrize("n,copies", [(24, 1), (64, 1), (64, 100), (300, 1), (300, 120), (600, 4), (1100, 32),
                                      (2047, 1)])
def test_small_components(engine, n, copies, path):
    # (components of few vertices: several, for the mean over as many)
    comps = [component(n, 7 * n + k) for k in range(max(1, 400 // n))]
    want = np.concatenate([exact(engine, c) for c in comps])
    g = engine.upload(comps * copies)
    got, st = g.run(path=path, precision=bcx.PREC_FP64)
    g.free()
    off = (got - np.tile(want, copies)) / np.spacing(np.tile(want, copies))
    rms = math.sqrt(float(np.mean(off ** 2)))
    print("n", n, "copies", copies, "path", path, "rms ulp", rms, flush=True)
    assert rms < BOUND, rms


@pytest.mark.parametrize("path", [bcx.PATH_PLAIN, bcx.PATH_BATCHED])
def test_sizes_beside_each_other(engine, path):
    """Components that leave four, two and no accumulators' room beside their waves
    (the launch's LDS is the largest one's), in tiles of up to 64 sources."""
    comps = [component(n, n + k) for n, m in ((64, 6), (300, 1), (640, 1), (900, 1), (1100, 1)) for k in range(m)]
    want = [exact(engine, c) for c in comps]
    g = engine.upload(comps * 30)
    got, _ = g.run(path=path, precision=bcx.PREC_FP64)
    g.free()
    got = got.reshape(30, -1)
    at = 0
    for n in (64, 300, 640, 900, 1100):
        w = np.concatenate([x for x in want if len(x) == n])
        off = (got[:, at:at + len(w)] - w) / np.spacing(w)
        at += len(w)
        rms = math.sqrt(float(np.mean(off ** 2)))
        print("n", n, "path", path, "rms ulp", rms, flush=True)
        assert rms < BOUND, (n, rms)


@pytest.mark.parametrize("n", [40, 98, 300, 1000])
def test_call_without_allocation(engine, n):
    comps = [component(n, 7 * n + k) for k in range(max(1, 800 // n))]
    want = np.concatenate([exact(engine, c) for c in comps])
    got = np.concatenate([noalloc(engine, c, None, bcx.PREC_FP64) for c in comps])
    rms = math.sqrt(float(np.mean(((got - want) / np.spacing(want)) ** 2)))
    print("no allocation: n", n, "rms ulp", rms, flush=True)
    assert rms < BOUND, rms


@pytest.mark.parametrize("path", [bcx.PATH_PLAIN, bcx.PATH_BATCHED])
@pytest.mark.parametrize("k", [64, 361, 1500])
def test_per_source_kernel(engine, k, path):
    """A grid of 3600 vertices, whose short rows are summed in one order by every
    run of the kernel: k of its sources."""
    w = 60
    edges = [(y * w + x, y * w + x + 1) for y in range(w) for x in range(w - 1)]
    edges += [(y * w + x, (y + 1) * w + x) for y in range(w - 1) for x in range(w)]
    c = bcx.Host.from_edges(w * w, edges).decompose(use_chains=False).components()[0]
    assert c.n == w * w and not np.any(c.reach)
    sub = np.sort(np.random.default_rng(k).permutation(c.n)[:k]).astype(np.int64)
    kw = dict(path=bcx.PATH_PLAIN, precision=bcx.PREC_FP64, use_chains=False)
    delta = np.array([engine.debug_source(c, int(s), **kw)[3] for s in sub])
    g = engine.upload([c])
    got, _ = g.run(path=path, precision=bcx.PREC_FP64, use_chains=False, subset=sub)
    g.free()
    want = np.array([math.fsum(delta[:, v]) for v in range(c.n)])
    pos = want > 0
    off = (got[pos] - want[pos]) / np.spacing(want[pos])
    rms = math.sqrt(float(np.mean(off ** 2)))
    print("k", k, "path", path, "rms ulp", rms, flush=True)
    assert rms < BOUND, rms


def dependencies(n, adj, s):
    """Dependencies of source s in extended precision."""
    level, order = {s: 0}, [s]
    sigma = np.zeros(n, np.longdouble)
    sigma[s] = 1
    for v in order:
        for w in adj[v]:
            if w not in level:
                level[w] = level[v] + 1
                order.append(w)
            if level[w] == level[v] + 1:
                sigma[w] += sigma[v]
    delta = np.zeros(n, np.longdouble)
    for v in reversed(order):
        for w in adj[v]:
            if level[w] == level[v] + 1:
                delta[v] += sigma[v] / sigma[w] * (1 + delta[w])
    delta[s] = 0
    return delta


def test_rows_of_the_per_source_kernel(engine):
    """Rows of 200 arcs, walked with a lane per arc: their sums are made of four
    parts of at most 64 terms, (0.25 64 / 3 + 1.5) squares of 0.32 ulp, the terms'
    own rounding is spread over 200, and the product with the count rounds once:
    0.9 ulp.  The bound is 1.3 times that (one part of 200: 2.6)."""
    rng = np.random.default_rng(11)
    A, B, C = 40, 300, 600
    n = 1 + A + B + C
    e = [(0, 1 + a) for a in range(A)]
    e += [(1 + a, 1 + A + int(b)) for a in range(A) for b in rng.choice(B, 200, replace=False)]
    e += [(1 + A + b, 1 + A + B + int(c)) for b in range(B) for c in rng.choice(C, 7, replace=False)]
    deg = np.bincount(np.array(e).ravel(), minlength=n)
    e += [(1 + A + c % B, 1 + A + B + c) for c in range(C) if deg[1 + A + B + c] == 0]
    adj = [[] for _ in range(n)]
    for a, b in sorted(set(e)):
        adj[a].append(b)
        adj[b].append(a)
    rp = np.concatenate([[0], np.cumsum([len(x) for x in adj])]).astype(np.int32)
    comp = bcx.HostComponent.from_csr(rp, np.concatenate(adj).astype(np.int32), np.zeros(n, np.int32))
    want = dependencies(n, adj, 0)[1:1 + A]
    got = engine.debug_source(comp, 0, path=bcx.PATH_PLAIN, precision=bcx.PREC_FP64)[3][1:1 + A]
    rms = math.sqrt(float(np.mean(((got - want) / np.spacing(want.astype(np.float64))) ** 2)))
    print("rows: rms ulp", rms, flush=True)
    assert rms < 1.2, rms
