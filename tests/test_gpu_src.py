"""The wave-per-source kernel of small components at the sizes where it can go
wrong: list and level-code words that are just full (63, 64, 65 vertices), the
smallest and largest component it takes (3 and 2048 vertices) and the first
that it leaves to the 64-source kernel, rows longer than a wave, path counts
past 64 bits, a deep cycle, and source counts around a tile's.  Whole-component
BC against the oracle on both paths: FP64 within 1e-9, FP32C within 1e-6
relative (the bars of the other kernels), zero BC exact."""
import numpy as np
import pytest

import bcx
import oracle
from helpers import relerr

pytestmark = pytest.mark.gpu


def ring_chords(n, m, seed):
    rng = np.random.default_rng(seed)
    e = {(min(i, (i + 1) % n), max(i, (i + 1) % n)) for i in range(n)}
    while len(e) < min(n + m, n * (n - 1) // 2):
        a, b = map(int, rng.integers(0, n, 2))
        if a != b:
            e.add((min(a, b), max(a, b)))
    return n, sorted(e)


def graph(kind):
    if kind == "triangle":
        return 3, [(0, 1), (1, 2), (0, 2)]
    if kind == "clique":  # rows of 89 arcs: a wave walks them
        return 90, [(a, b) for a in range(90) for b in range(a + 1, 90)]
    if kind == "wheel":  # one row of 700 arcs, counts through it
        return 701, [(i, (i + 1) % 700) for i in range(700)] + [(i, 700) for i in range(700)]
    if kind == "grid":  # corner counts C(88, 44) pass 2^64
        w = 45
        return w * w, [(y * w + x, y * w + x + 1) for y in range(w) for x in range(w - 1)] + \
            [(y * w + x, (y + 1) * w + x) for y in range(w - 1) for x in range(w)]
    if kind == "cycle":
        return 1501, [(i, (i + 1) % 1501) for i in range(1501)]
    n, m = {"n63": (63, 60), "n64": (64, 60), "n65": (65, 60), "n2047": (2047, 6000), "n2048": (2048, 6000),
            "n2048 dense": (2048, 14000)}[kind]
    return ring_chords(n, m, n + m)


@pytest.mark.parametrize("kind", ["triangle", "n63", "n64", "n65", "clique", "wheel", "grid", "cycle", "n2047",
                                  "n2048", "n2048 dense"])
def test_component(engine, kind):
    n, e = graph(kind)
    c = bcx.Host.from_edges(n, e).decompose().components()[0]
    assert c.n == n
    rng = np.random.default_rng(n)
    g = engine.upload([c])
    try:
        for k in (n, 1, 16, 17, 65):
            sub = None if k == n else np.sort(rng.choice(n, size=min(k, n), replace=False))
            want = oracle.component_bc(c.row_ptr, c.col, c.reach,
                                       sources=None if sub is None else sub.astype(np.int32))
            for path, prec, tol in ((bcx.PATH_PLAIN, bcx.PREC_FP64, 1e-9), (bcx.PATH_BATCHED, bcx.PREC_FP64, 1e-9),
                                    (bcx.PATH_BATCHED, bcx.PREC_FP32C, 1e-6)):
                got, st = g.run(path=path, precision=prec, subset=sub)
                mx, _, zeros = relerr(got, want)
                assert mx < tol and zeros, (kind, k, path, prec, mx)
                if kind == "grid" and k == n:
                    assert st["n_f64_sigma"] > 0
    finally:
        g.free()
