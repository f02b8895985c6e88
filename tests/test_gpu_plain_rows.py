"""The per-source kernel's row walks and launch shapes at their edges: rows
just at and above the lane walk's and the wave walk's lengths (8, 9, 256, 257
arcs), components at the sizes where the waves per source change (8192 and
49152 vertices) and where the level codes leave LDS (400000), more levels than
the LDS offsets hold, and FP64 counts on long rows.  BC of sampled sources
against the oracle, 1e-9 relative, zero BC exact."""
import numpy as np
import pytest

import bcx
import oracle
from helpers import relerr

pytestmark = pytest.mark.gpu


def csr(n, e):
    e = np.asarray(e, np.int64)
    src = np.concatenate([e[:, 0], e[:, 1]])
    dst = np.concatenate([e[:, 1], e[:, 0]])
    order = np.argsort(src, kind="stable")
    rp = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))])
    return bcx.HostComponent.from_csr(rp, dst[order].astype(np.int32),
                                      reach=np.arange(n, dtype=np.int32) % 3)


def ring(n, chords, seed):
    rng = np.random.default_rng(seed)
    v = np.arange(n)
    e = np.concatenate([np.stack([v, (v + 1) % n], 1), rng.integers(0, n, size=(chords, 2))])
    e = e[e[:, 0] != e[:, 1]]
    _, first = np.unique(e.min(1) * n + e.max(1), return_index=True)
    return e[np.sort(first)]


def hubs(n, degrees):
    """A ring whose first vertices have exactly the given degrees."""
    e = [(i, (i + 1) % n) for i in range(n)]
    at = len(degrees) + 2
    for h, d in enumerate(degrees):
        for _ in range(d - 2):
            e.append((h, at))
            at += 1
    assert at < n
    return e


@pytest.mark.parametrize("degrees", [[8], [9], [8, 9, 256], [257], [9, 256, 257, 600]])
@pytest.mark.parametrize("log2", [0, 6])
def test_row_lengths(engine, degrees, log2):
    n = 3001
    c = csr(n, hubs(n, degrees))
    sub = np.unique(np.concatenate([np.arange(8), np.linspace(8, n - 1, 20).astype(np.int64)]))
    want = oracle.component_bc(c.row_ptr, c.col, c.reach, sources=sub.astype(np.int32))
    (got,), st = engine.bc([c], subset=sub, sigma_threshold_log2=log2)
    mx, _, zeros = relerr(got, want)
    assert mx < 1e-9 and zeros, (degrees, log2, mx)


@pytest.mark.parametrize("n", [2049, 8192, 8193, 49152, 49153, 400000, 400001])
def test_sizes(engine, n):
    c = csr(n, ring(n, 2 * n, n))
    sub = np.linspace(0, n - 1, 9).astype(np.int64)
    want = oracle.component_bc(c.row_ptr, c.col, c.reach, sources=sub.astype(np.int32), threads=9)
    (got,), st = engine.bc([c], subset=sub)
    mx, _, zeros = relerr(got, want)
    assert mx < 1e-9 and zeros, (n, mx)
    (got,), st = engine.bc([c], subset=sub, sigma_threshold_log2=3)  # FP64 counts
    assert st["n_f64_sigma"] > 0
    mx, _, zeros = relerr(got, want)
    assert mx < 1e-9 and zeros, (n, mx)


@pytest.mark.parametrize("n", [4099, 400003])
def test_deep(engine, n):
    """A cycle of n vertices beside chords over its first 100: more than 1024
    levels, chain sources included."""
    m = 5000 if n > 10000 else n  # the deep part; the rest is bushy
    e = [(i, (i + 1) % m) for i in range(m)] + [(0, 50), (20, 90)]
    if n > m:
        e += [(m + i, int(x)) for i, x in enumerate(np.random.default_rng(1).integers(0, 100, n - m))]
        e += [(m + i, 100 + (i % 7)) for i in range(n - m)]
    host = bcx.Host.from_edges(n, np.asarray(e, np.int32)).decompose()
    c = max(host.components(), key=lambda c: c.n)
    assert c.n_chains > 0
    sub = np.unique(np.concatenate([np.linspace(0, c.n - 1, 6).astype(np.int64), c.chain_nodes[[0, 700, -1]]]))
    want = oracle.component_bc(c.row_ptr, c.col, c.reach, sources=sub.astype(np.int32), threads=9)
    for chains in (True, False):
        (got,), st = engine.bc([c], subset=sub, use_chains=chains)
        assert st["max_level"] > 1024
        mx, _, zeros = relerr(got, want)
        assert mx < 1e-9 and zeros, (n, chains, mx)


@pytest.mark.parametrize("n,chords", [(2500, 100), (2500, 3750), (2500, 3760), (20000, 900), (20001, 900)])
@pytest.mark.parametrize("prec", [bcx.PREC_FP64, bcx.PREC_FP32C])
def test_dependencies_in_vertex_order(engine, n, chords, prec):
    """Sparse components up to 20000 vertices and 5 arcs per vertex add a
    source's dependencies in vertex order; one over either line adds them one by
    one.  Ragged source lists, the whole list twice (rows are used again)."""
    c = csr(n, ring(n, chords, n + chords))
    sub = np.unique(np.linspace(0, n - 1, 601).astype(np.int64))
    want = oracle.component_bc(c.row_ptr, c.col, c.reach, sources=sub.astype(np.int32))
    path = bcx.PATH_PLAIN if prec == bcx.PREC_FP64 else bcx.PATH_BATCHED
    tol = 1e-9 if prec == bcx.PREC_FP64 else 1e-6
    for _ in range(2):
        (got,), st = engine.bc([c], subset=sub, path=path, precision=prec, flags=bcx.FLAG_NO_TUNE)
        mx, _, zeros = relerr(got, want)
        assert mx < tol and zeros, (n, chords, prec, mx)


@pytest.mark.parametrize("spare", [2, 8, 400])
def test_little_room_beside_the_rows(engine, spare):
    """A capacity that holds the workgroups' rows and `spare` MiB: the run takes
    what fits of the ordered copy and the split accumulators, and is never
    refused for them.  Every vertex of a bipartite graph of 40 hubs."""
    rng = np.random.default_rng(spare)
    n, hubs_n = 5000, 40
    e = [(h, v) for v in range(hubs_n, n) for h in rng.choice(hubs_n, size=3, replace=False)]
    c = csr(n, e)
    sub = np.sort(rng.permutation(n)[:700]).astype(np.int64)
    rows = ((n + 2 + 63) // 64 * 64) * 28 * min(len(sub), 2 * engine.info()[0])
    eng = bcx.Engine(0, mem_cap=rows + (spare << 20))
    (got,), st = eng.bc([c], subset=sub)
    eng.close()
    want = oracle.component_bc(c.row_ptr, c.col, c.reach, sources=sub.astype(np.int32))
    mx, _, zeros = relerr(got, want)
    assert mx < 1e-9 and zeros, mx
