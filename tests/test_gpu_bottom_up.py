"""Multi-launch tiles whose levels are found bottom-up (from a frontier of more
than a sixteenth of the vertices) beside levels that are pushed, against the
oracle source by source: a narrow ladder into a random core (the frontier
crosses the line on the way), two hubs above the slice threshold, contracted
chains with sources inside them, ragged and full tiles of every width, integer
and FP64 path counts."""
import numpy as np
import pytest

import bcx
from tilecheck import check_tile

pytestmark = pytest.mark.gpu

MULTI = bcx.FLAG_NO_SMALL_KERNEL | bcx.FLAG_NO_WG_KERNEL


def _simple(e):
    return sorted({(min(a, b), max(a, b)) for a, b in ((int(a), int(b)) for a, b in e) if a != b})


def _graph(seed):
    rng = np.random.default_rng(seed)
    core, rungs = 900, 40
    e = [tuple(x) for x in rng.integers(0, core, size=(2200, 2)) if x[0] != x[1]]
    e += [(i, i + 1) for i in range(core - 1)]
    e += [(0, v) for v in range(2, 620)] + [(5, v) for v in range(100, 640)]  # hubs
    n = core
    for r in range(rungs):  # ladder, one end on the core
        a, b = n + 2 * r, n + 2 * r + 1
        e.append((a, b))
        if r:
            e += [(a - 2, a), (b - 2, b)]
    e += [(n, 7), (n + 1, 333)]
    n += 2 * rungs
    for q in range(30):  # chains between core vertices, one of them at a hub
        ends = (5 if q == 0 else int(rng.integers(0, core)), int(rng.integers(0, core)))
        k = int(rng.integers(1, 9))
        path = [ends[0], *range(n, n + k), ends[1]]
        e += list(zip(path[:-1], path[1:]))
        n += k
    return n, _simple(e)


@pytest.mark.parametrize("spl", [1, 2, 4])
@pytest.mark.parametrize("width", [1, 63, 64])
def test_bottom_up_levels(engine, spl, width):
    n, e = _graph(10 * spl + width)
    c = max(bcx.Host.from_edges(n, e).decompose(use_chains=True).components(), key=lambda c: c.n)
    ns = 1 if width == 1 else 64 * (spl - 1) + width
    rng = np.random.default_rng(spl)
    far = [c.n - 1 - i for i in range(min(ns, 40))]  # (ladder and chain vertices among them)
    rest = rng.permutation(c.n - 40)[:ns - len(far)]
    srcs = np.concatenate([far, rest]).astype(np.int32)
    for prec in (bcx.PREC_FP64, bcx.PREC_FP32C):
        check_tile(engine, c, srcs, prec, MULTI, bcx.KERNEL_MULTI, want_f64=False, tag=f"up/{spl}/{width}", spl=spl)


@pytest.mark.parametrize("spl", [1, 4])
def test_bottom_up_fp64_counts(engine, spl):
    """Complete layers of 3, then a wide layer: path counts beyond 64 bits
    before the frontier widens; FP64 counts in the oracle's order."""
    L, k, wide = 60, 3, 700
    e = [(i * k + a, (i + 1) * k + b) for i in range(L - 1) for a in range(k) for b in range(k)]
    n = L * k
    rng = np.random.default_rng(spl)
    e += [((L - 1) * k + a, n + w) for w in range(wide) for a in range(k)]
    e += [(n + int(a), n + int(b)) for a, b in rng.integers(0, wide, size=(1500, 2)) if a != b]
    c = max(bcx.Host.from_edges(n + wide, _simple(e)).decompose(use_chains=False).components(), key=lambda c: c.n)
    srcs = np.arange(64 * spl) * (c.n // (64 * spl))
    check_tile(engine, c, srcs.astype(np.int32), bcx.PREC_FP32C, MULTI, bcx.KERNEL_MULTI, tag=f"up64/{spl}", spl=spl)
