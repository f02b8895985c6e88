"""A component whose sources do not reach every vertex (uploaded as it is; the
decomposition makes none) on the plain path: what a source does not reach gets
nothing from it.  (The batched path orders its sources by breadth-first search
and wants components connected, as bcx_component says.)  Two rings with chords
side by side, each part against the oracle on its own."""
import numpy as np
import pytest

import bcx
import oracle
from helpers import relerr

pytestmark = pytest.mark.gpu


def ring(n, chords, seed):
    rng = np.random.default_rng(seed)
    e = np.concatenate([np.stack([np.arange(n), (np.arange(n) + 1) % n], 1), rng.integers(0, n, size=(chords, 2))])
    e = np.sort(e[e[:, 0] != e[:, 1]], axis=1)
    return np.unique(e, axis=0).astype(np.int32)


def with_chains(e, n, k):
    """e and k paths of three vertices between vertices of it."""
    ends = np.random.default_rng(k).choice(n, size=(k, 2), replace=False)
    out, nodes = [e], []
    for i, (a, b) in enumerate(ends):
        v = n + 3 * i
        out.append(np.asarray([(a, v), (v, v + 1), (v + 1, v + 2), (v + 2, b)], np.int32))
        nodes.append([v, v + 1, v + 2])
    return np.concatenate(out), n + 3 * k, ends, np.asarray(nodes)


def component(sizes, chains):
    parts, ends, nodes, off = [], [], [], 0
    for i, n in enumerate(sizes):
        e, m, en, no = with_chains(ring(n, n // 2, i), n, chains)
        parts.append((off, m, e))
        ends.append(en + off)
        nodes.append(no + off)
        off += m
    rp, col = oracle.csr_from_edges(off, np.concatenate([e + o for o, _, e in parts]))
    reach = np.random.default_rng(1).integers(0, 5, off).astype(np.int32)
    ends, nodes = np.concatenate(ends), np.concatenate(nodes)
    c = bcx.HostComponent.from_csr(rp, col, reach, np.arange(0, 3 * len(ends) + 1, 3, dtype=np.int32),
                                   nodes.reshape(-1).astype(np.int32), ends.reshape(-1).astype(np.int32))
    return c, parts, reach


def exact(c, parts, reach, sub):
    want = np.zeros(c.n)
    for off, n, e in parts:
        s = sub[(sub >= off) & (sub < off + n)] - off
        rp, col = oracle.csr_from_edges(n, e)
        want[off:off + n] = oracle.component_bc(rp, col, reach[off:off + n], sources=s.astype(np.int32), threads=16)
    return want


PLAIN = dict(path=bcx.PATH_PLAIN)
ROWS = dict(PLAIN, row_cap_bytes=1 << 30)


@pytest.mark.parametrize("sizes,kw,tol", [((2000, 900), PLAIN, 1e-9), ((300, 6000), PLAIN, 1e-9),
                                          ((2000, 900), ROWS, 1e-9), ((300, 6000), ROWS, 1e-9), ((40, 60), ROWS, 1e-9),
                                          ((2000, 900), dict(ROWS, sigma_threshold_log2=3), 1e-9),
                                          ((40, 60), PLAIN, 1e-9)])
def test_parts(engine, sizes, kw, tol):
    c, parts, reach = component(sizes, 20)
    want = exact(c, parts, reach, np.arange(c.n))
    g = engine.upload([c])
    try:
        for _ in range(2):
            got, _ = g.run(**kw)
            mx, _, zeros = relerr(got, want)
            assert mx < tol and zeros, mx
    finally:
        g.free()


def test_levels_of_one_source(engine):
    """The probe of a source reports what it does not reach as it always has."""
    c, parts, _ = component((2000, 900), 20)
    for src in (3, parts[1][0] + 5):
        lv, su, _, dl, f64 = engine.debug_source(c, src)
        own = next(p for p in parts if p[0] <= src < p[0] + p[1])
        out = np.ones(c.n, bool)
        out[own[0]:own[0] + own[1]] = False
        assert np.all(lv[out] == 2 ** 31 - 1) and np.all(su[out] == 0) and np.all(dl[out] == 0)
        assert np.all(lv[~out] < c.n) and np.all(su[~out] > 0)
