"""Which kernel a batched component runs on never shows in its FP32C result.

Every kernel but the multi-launch tiles rounds the same terms to FP32 at the same
points and sums them in the same order (1e-12 apart: FP64 rounding of the
accumulated BC); those tiles contract chains and slice the rows of hubs (1e-10
to 7e-9 apart).  So a component runs on them in every call or in none, and
counts past 64 bits turn the same 64 sources to FP64 terms on whichever kernel
they are met.
"""
import time

import numpy as np
import pytest

import bcx

pytestmark = pytest.mark.gpu

B, F32 = bcx.PATH_BATCHED, bcx.PREC_FP32C
SAME = 1e-12


def giant(cfg, scale, seed=3):
    n, uv = bcx.generate(cfg, 0, scale)
    uv = np.random.default_rng(seed).permutation(n).astype(np.int32)[uv]
    return max(bcx.Host.from_edges(n, uv).decompose().components(), key=lambda c: c.n)


def far(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


ROWS, SLICED = bcx.FLAG_WG_KERNEL, bcx.FLAG_NO_WG_KERNEL


@pytest.mark.parametrize("cfg,scale,chains,flags", [
    (2, 0.022, True, ROWS), (2, 0.022, False, ROWS), (5, 0.06, True, ROWS), (5, 0.06, False, ROWS),
    (2, 0.047, True, SLICED), (2, 0.05547, True, SLICED), (2, 0.05547, False, SLICED), (2, 0.0555, True, ROWS),
    (2, 0.08, True, ROWS), (2, 0.08, False, ROWS), (5, 0.17, True, SLICED), (2, 0.12, True, SLICED),
    (2, 0.12, False, ROWS)])
def test_fp32c_does_not_depend_on_the_number_of_sources(engine, cfg, scale, chains, flags):
    """Power-law cores of 18.6k to 101k vertices and R-MAT cores: subsets of every
    size, with the tuner's rates of each, equal the kernel that the flags force,
    which is the one that full jobs of the component were given before the
    per-source kernel was there (two cores of 46.7k: tiles over the last sources
    that were sampled)."""
    c = giant(cfg, scale)
    order = np.random.default_rng(7).permutation(c.n).astype(np.int64)
    g = engine.upload([c])
    try:
        for k in (64, 600, 4096, 20000):
            kw = dict(path=B, precision=F32, subset=order[:k], use_chains=chains)
            got, st = g.run(**kw)
            want, _ = g.run(flags=flags, **kw)
            print("case", cfg, scale, c.n, k, "multi", st["n_comp_multi"], "contracted", st["n_contracted"],
                  far(got, want), flush=True)
            assert far(got, want) < SAME
    finally:
        g.free()


def test_per_source_runs_are_told_apart(engine):
    """The per-source kernel runs where it should: deep and mid-size components
    in either precision, not where a flag or a lane width asks for tiles, nor
    where an FP32C run met an overflow and went to the tiles."""
    c = giant(2, 0.006)
    g = engine.upload([c])
    try:
        for kw, want in ((dict(precision=F32), 1), (dict(precision=bcx.PREC_FP64), 1),
                         (dict(precision=F32, flags=bcx.FLAG_WG_KERNEL), 0), (dict(precision=F32, sources_per_lane=2), 0),
                         (dict(precision=bcx.PREC_FP64, sigma_threshold_log2=6), 1),
                         (dict(precision=F32, sigma_threshold_log2=6), 0)):
            _, st = g.run(path=B, subset=np.arange(64), **kw)
            assert st["n_comp_wg"] == 1 and engine.run_by_source() == want, (kw, want)
    finally:
        g.free()


@pytest.mark.parametrize("prec", [bcx.PREC_FP64, F32])
@pytest.mark.parametrize("width_first", [False, True])
def test_lane_width_is_kept_and_keeps_nothing(engine, prec, width_first):
    """A run that fixes the sources per lane gets tiles of that width, whatever
    earlier runs of the component measured, and leaves no choice behind for
    those that do not (a 17k grid: source by source)."""
    c = giant(4, 0.23)
    assert c.n >= 16384
    sub = np.arange(0, c.n, 67)
    g = engine.upload([c])
    try:
        seen = []
        for width in ([1, 0, 1, 0] if width_first else [0, 1, 0, 1]):
            bc, st = g.run(path=B, precision=prec, subset=sub, sources_per_lane=width)
            seen.append(bc)
            assert engine.run_by_source() == (0 if width else 1), (width, st)
            assert not width or st["n_comp_wg"] == 1 or st["sched_sources_per_lane"] == width
        for bc in seen[1:]:
            assert far(bc, seen[0]) < SAME
    finally:
        g.free()


def test_precisions_are_measured_apart(engine):
    """Counts that leave 64 bits end FP32C's per-source runs of a component, not
    those with FP64 terms, in either order; the overflow is met once."""
    c = giant(4, 0.035, 0)
    sub = np.arange(0, c.n, 2)
    for order in ((F32, bcx.PREC_FP64), (bcx.PREC_FP64, F32)):
        g = engine.upload([c])
        try:
            for prec in order + order:
                g.run(path=B, precision=prec, subset=sub)
                assert engine.run_by_source() == (prec == bcx.PREC_FP64)
        finally:
            g.free()


def test_first_call_on_a_mid_size_core(engine):
    """The first run of a 23k R-MAT core takes the samples that its choice of
    kernel needs; only a run that asks for the multi-launch tiles, and a core
    above the line, pays for a tuned schedule (six candidates twice)."""
    c = giant(5, 0.06)
    g = engine.upload([c])
    kw = dict(path=B, subset=np.arange(64))
    g.run(**kw)  # (code objects, buffers)
    g.free()
    took = {}
    for flags in (0, bcx.FLAG_NO_WG_KERNEL):
        g = engine.upload([c])
        try:
            t = time.perf_counter()
            g.run(flags=flags, **kw)
            took[flags] = time.perf_counter() - t
        finally:
            g.free()
    print("case first call", {k: round(1e3 * v, 1) for k, v in took.items()}, flush=True)
    assert took[0] < 0.6 * took[bcx.FLAG_NO_WG_KERNEL]


@pytest.mark.parametrize("cfg,scale,seed,bits", [(4, 0.035, 0, 0), (4, 0.035, 2, 0), (4, 0.03, 5, 0),
                                                 (2, 0.006, 3, 8), (2, 0.006, 3, 9)])
def test_the_same_sources_turn_to_fp64(engine, cfg, scale, seed, bits):
    """Components with counts past 64 bits (or a forced limit) from some sources
    only: the sources that get FP64 terms are those of the workgroup kernel's
    tiles, whether the counts were foreseen (grids whose hub's counts, by the
    numbering, reach 2^43, 2^59 and 2^48) or met by a per-source run."""
    c = giant(cfg, scale, seed)
    assert c.n > 2048
    sub = np.random.default_rng(11).permutation(c.n)[:2000].astype(np.int64)
    g = engine.upload([c])
    try:
        kw = dict(path=B, precision=F32, subset=sub, sigma_threshold_log2=bits)
        got = [g.run(**kw) for _ in range(2)]
        want, ws = g.run(flags=bcx.FLAG_WG_KERNEL, **kw)
        for bc, st in got:
            print("case", cfg, scale, c.n, bits, "FP64", ws["n_f64_sigma"], st["n_f64_sigma"], far(bc, want), flush=True)
            assert st["n_f64_sigma"] == ws["n_f64_sigma"] and far(bc, want) < SAME
    finally:
        g.free()
