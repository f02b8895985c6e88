"""Components of the batched path whose sources run one by one (the per-source
kernel in the run's precision): FP64 and FP32C against the oracle and against
the workgroup kernel's tiles.  FP32C rounds the same terms at the same points
and sums them in the same order on both, so the two differ by FP64 rounding of
the accumulated BC alone (a few thousand terms: under 1e-12)."""
import numpy as np
import pytest

import bcx
import oracle
from helpers import relerr

pytestmark = pytest.mark.gpu

B = bcx.PATH_BATCHED


def component(kind):
    if kind == "grid":  # counts past 2^64: FP64 from the start
        w = 60
        n, e = w * w, [(y * w + x, y * w + x + 1) for y in range(w) for x in range(w - 1)] + \
            [(y * w + x, (y + 1) * w + x) for y in range(w - 1) for x in range(w)]
    elif kind == "wheel":  # a row of 2999 arcs and rows of 3
        n, e = 3000, [(i, (i + 1) % 2999) for i in range(2999)] + [(i, 2999) for i in range(2999)]
    else:  # power law with hubs and chains
        n, e = bcx.generate(2, 0, 0.006)
    return max(bcx.Host.from_edges(n, np.asarray(e, np.int32)).decompose().components(), key=lambda c: c.n)


@pytest.mark.parametrize("kind", ["grid", "wheel", "power law"])
@pytest.mark.parametrize("log2", [0, 6])
def test_single(engine, kind, log2):
    c = component(kind)
    assert c.n > 2048
    g = engine.upload([c])
    try:
        for k in ([c.n] if kind == "power law" else []) + [257, 1]:  # (5080 sources: split accumulator)
            sub = np.linspace(0, c.n - 1, k).astype(np.int64) if k > 1 else np.array([c.n // 2])
            want = oracle.component_bc(c.row_ptr, c.col, c.reach, sources=np.unique(sub).astype(np.int32), threads=16)
            for prec, tol in ((bcx.PREC_FP64, 1e-9), (bcx.PREC_FP32C, 1e-6)):
                got, st = g.run(path=B, precision=prec, subset=sub, sigma_threshold_log2=log2)
                mx, _, zeros = relerr(got, want)
                assert mx < tol and zeros, (kind, k, prec, mx)
                assert st["n_comp_wg"] == 1
                tiles, _ = g.run(path=B, precision=prec, subset=sub, sigma_threshold_log2=log2,
                                 flags=bcx.FLAG_WG_KERNEL)
                mx, _, _ = relerr(got, tiles)
                assert mx < 1e-12, (kind, k, prec, mx)
    finally:
        g.free()
