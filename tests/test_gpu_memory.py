"""Batched runs under a memory cap: the per-source kernel's rows are an option,
so a job that the tiles alone have room for is never refused for them."""
import numpy as np
import pytest

import bcx
import oracle
from helpers import relerr

pytestmark = pytest.mark.gpu

B = bcx.PATH_BATCHED


def giant(cfg, scale):
    n, uv = bcx.generate(cfg, 0, scale)
    return max(bcx.Host.from_edges(n, uv).decompose().components(), key=lambda c: c.n)


def rows(engine, c, sources):
    """Bytes of the rows that a per-source run takes at least."""
    return (c.n + 2 + 63) // 64 * 64 * 28 * min(sources, 2 * engine.info()[0])


def slot(c):
    """Bytes of a multi-launch tile in flight, about."""
    return c.n * 4 * (8 + 24 + 512 + 512 + 96)


def check(g, c, sub, tol, **kw):
    got, st = g.run(path=B, subset=sub, **kw)
    want = oracle.component_bc(c.row_ptr, c.col, c.reach, sources=sub.astype(np.int32), threads=16)
    mx, _, zeros = relerr(got, want)
    assert mx < tol and zeros, mx
    return st


@pytest.mark.parametrize("prec,tol", [(bcx.PREC_FP64, 1e-9), (bcx.PREC_FP32C, 1e-6)])
def test_first_run_of_few_sources(engine, prec, tol):
    """An 18.6k core, 64 sources first, under a cap with room for two tiles in
    flight and the rows of 64 sources, not for those of the tuner's sample."""
    c = giant(2, 0.022)
    assert c.n >= 16384
    cap = 2 * slot(c) + rows(engine, c, 64)
    assert cap < rows(engine, c, c.n) + slot(c)
    eng = bcx.Engine(0, mem_cap=cap)
    try:
        g = eng.upload([c])
        for k in (64, 700):
            check(g, c, np.linspace(0, c.n - 1, k).astype(np.int64), tol, precision=prec)
        g.free()
    finally:
        eng.close()


def test_rows_make_room_for_tiles(engine):
    """A cap with room for a deep component's rows or one tile in flight, not
    both: source by source, then on the tiles, then as there is room."""
    c = giant(4, 0.23)
    assert c.n >= 16384
    eng = bcx.Engine(0, mem_cap=rows(engine, c, c.n) + slot(c) // 2 + (16 << 20))
    sub = np.linspace(0, c.n - 1, 600).astype(np.int64)
    try:
        g = eng.upload([c])
        for flags in (0, bcx.FLAG_NO_WG_KERNEL | bcx.FLAG_NO_TUNE, bcx.FLAG_NO_TUNE):
            check(g, c, sub, 1e-9, flags=flags)
            assert flags or eng.run_by_source() == 1
        g.free()
    finally:
        eng.close()


def test_tiles_and_rows_in_one_run(engine):
    """Two components, one for the tiles and one for the per-source kernel, under
    a cap that the tiles fill: the other goes to the tiles as well."""
    a, b = giant(5, 0.12), giant(4, 0.2)
    eng = bcx.Engine(0, mem_cap=int(1.15 * slot(a)) + rows(engine, b, b.n) // 2 + (20 << 20))
    sub = np.concatenate([np.linspace(0, a.n - 1, 64).astype(np.int64), a.n + np.linspace(0, b.n - 1, 600).astype(np.int64)])
    try:
        g = eng.upload([a, b])
        got, _ = g.run(path=B, subset=sub, flags=bcx.FLAG_NO_TUNE)
        g.free()
    finally:
        eng.close()
    for c, off, s in ((a, 0, sub[:64]), (b, a.n, sub[64:] - a.n)):
        want = oracle.component_bc(c.row_ptr, c.col, c.reach, sources=s.astype(np.int32), threads=16)
        mx, _, zeros = relerr(got[off:off + c.n], want)
        assert mx < 1e-9 and zeros, mx


def test_run_after_one_that_failed(engine):
    """A run whose result download finds no room is refused after its kernel was
    started; the next run of the context is not disturbed by what was queued."""
    rng = np.random.default_rng(5)
    comps = []
    for i in range(40):
        n = 100 + i
        e = np.concatenate([np.stack([np.arange(n), (np.arange(n) + 1) % n], 1), np.stack([np.arange(n), (np.arange(n) + 2 + i % 7) % n], 1)])
        e = np.unique(np.sort(e, axis=1), axis=0)
        rp, col = oracle.csr_from_edges(n, e[rng.permutation(len(e))])
        comps.append(bcx.HostComponent.from_csr(rp, col, rng.integers(0, 5, n).astype(np.int32)))
    want = np.concatenate([oracle.component_bc(c.row_ptr, c.col, c.reach) for c in comps])
    sub = np.arange(comps[0].n, len(want))  # (every component but the first)

    def runs(cap):
        eng = bcx.Engine(0, mem_cap=cap)
        try:
            eng.bc(comps, path=B)
            return True
        except bcx.BcxError as e:
            assert e.code == -4
            return False
        finally:
            eng.close()

    lo, hi = 1 << 12, 1 << 22
    while hi - lo > 256:  # the least cap that a whole run fits in
        lo, hi = ((lo + hi) // 2, hi) if not runs((lo + hi) // 2) else (lo, (lo + hi) // 2)
    eng = bcx.Engine(0, mem_cap=hi)
    try:
        g = eng.upload(comps)
        g.run(path=B)
        for _ in range(3):
            with pytest.raises(bcx.BcxError) as e:
                g.run(path=B, subset=sub)
            assert e.value.code == -4
            got, _ = g.run(path=B)
            mx, _, zeros = relerr(got, want)
            assert mx < 1e-9 and zeros, mx
        g.free()
    finally:
        eng.close()


def test_several_accumulators_make_room(engine):
    """FP64 runs of small components take several accumulators; a cap that holds a
    large component's rows, beside one accumulator alone, still does."""
    n, k = 700, 4
    e = np.concatenate([np.stack([np.arange(n), (np.arange(n) + s) % n], 1) for s in (1, 2, 9)])
    rp, col = oracle.csr_from_edges(n, e)
    small = bcx.HostComponent.from_csr(rp, col, np.zeros(n, np.int32))
    one = oracle.component_bc(small.row_ptr, small.col, small.reach)
    big = giant(4, 0.05)
    sub = np.linspace(0, big.n - 1, 300).astype(np.int64)
    part = oracle.component_bc(big.row_ptr, big.col, big.reach, sources=sub.astype(np.int32), threads=16)
    eng = bcx.Engine(0, mem_cap=rows(engine, big, 300) + 800000)
    assert 16 * 8 * (k * n + big.n) > 800000
    try:
        g = eng.upload([small] * k)
        got, _ = g.run(path=B)
        mx, _, zeros = relerr(got, np.tile(one, k))
        assert mx < 1e-9 and zeros, mx
        g.free()
        g = eng.upload([small] * k + [big])
        got, _ = g.run(path=bcx.PATH_PLAIN, subset=np.concatenate([np.arange(n), k * n + sub]))
        mx, _, zeros = relerr(got, np.concatenate([one, np.zeros((k - 1) * n), part]))
        assert mx < 1e-9 and zeros, mx
        g.free()
    finally:
        eng.close()
