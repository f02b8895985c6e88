"""Workloads that stand for the use of this framework: exact betweenness
centrality through its public entry points (`Engine.host_bc`, `DGraph.run`,
`bcx_bc_small_noalloc`), from graphs of two dozen vertices to cores of more than
a hundred and fifty thousand, on both paths and in both precisions.

Graphs come from the framework's own generators (the five benchmark
workloads at smaller scales) or are a ring with random chords.  A case is a
dict of plain values:

  entry      "host"    host_bc: a reduced graph on the host -> BC per vertex
                       (upload, run and free in every call)
             "run"     DGraph.run: components uploaded once, run many times
             "device"  bcx_bc_small_noalloc: one component in device memory
  graph      ring | blocks | mixed | many | grid | rmat
  n, degree  (ring) vertices, average degree
  scale      (the others) share of the workload's full size
  path, precision, chains   as in bcx_opts
  sources    0: every vertex, else that many vertices of the largest component
  pick       "random": drawn uniformly (the sampled mode of the command line),
             "tiles": runs of 256 in the library's order (a slice of a full job)
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "centrality-gpu_amd"))
import bcx  # noqa: E402

PATHS = {"plain": bcx.PATH_PLAIN, "batched": bcx.PATH_BATCHED}
PRECISIONS = {"fp64": bcx.PREC_FP64, "fp32c": bcx.PREC_FP32C}
WORKLOADS = {"blocks": 1, "mixed": 2, "many": 3, "grid": 4, "rmat": 5}


def listed():
    def case(name, entry, graph, path, precision, **kw):
        return {"name": name, "entry": entry, "graph": graph, "path": path, "precision": precision,
                "chains": True, "sources": 0, "pick": "random", **kw}

    return [
        # the smallest call: a graph of the size of the sample inputs, default
        # options, one shot; latency and launches are all there is
        case("ring_host_plain", "host", "ring", "plain", "fp64", n=24, degree=3.0),
        # a small analysis job with default options: 16 blocks joined at cut
        # vertices, a fifth of the edges chains, every source
        case("blocks_run_plain", "run", "blocks", "plain", "fp64", scale=1.0),
        # the same job on the batched path, as a user in a hurry runs it
        case("blocks_run_fp32c", "run", "blocks", "batched", "fp32c", scale=1.0),
        # a quarter of that job in one shot from the reduced host graph
        case("blocks_host_fp64", "host", "blocks", "batched", "fp64", scale=0.25),
        # a graph that falls apart into hundreds of small blocks beside one
        # larger core, every source
        case("many_run_fp32c", "run", "many", "batched", "fp32c", scale=0.01),
        # a power-law core with chains: a slice of a full job in whole tiles
        case("mixed_run_fp32c", "run", "mixed", "batched", "fp32c", scale=0.2, sources=6144, pick="tiles"),
        # the same kind of graph in the sampled mode: an odd number of sources
        # drawn uniformly, full precision
        case("mixed_run_fp64", "run", "mixed", "batched", "fp64", scale=0.2, sources=2001),
        # a denser, more skewed core (R-MAT): a slice of a full job
        case("rmat_run_fp32c", "run", "rmat", "batched", "fp32c", scale=0.25, sources=6144, pick="tiles"),
        # a deep, narrow graph whose path counts leave 64 bits: whole tiles
        case("grid_run_fp32c", "run", "grid", "batched", "fp32c", scale=0.35, sources=16384, pick="tiles"),
        # per-source default path on a power-law core, a sample of its sources
        case("mixed_run_plain", "run", "mixed", "plain", "fp64", scale=0.1, sources=1000),
        # per-source default path on a deep graph (FP64 path counts)
        case("grid_run_plain", "run", "grid", "plain", "fp64", scale=0.25, sources=2049),
        # a serving loop that may not allocate: one component in device memory
        case("ring_device_fp64", "device", "ring", "batched", "fp64", n=1000, degree=8.0),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    c = dict(rng.choice(listed()))
    del c["name"]
    c["chains"] = rng.random() < 0.8
    if c["graph"] == "ring":
        c["n"] = int(_log(rng, 5, 2048 if c["entry"] == "device" else 400))
        c["degree"] = round(min(rng.uniform(2.5, 10.0), (c["n"] - 1) / 2), 2)
        c["precision"] = rng.choice(["fp64", "fp32c"]) if c["entry"] == "device" else "fp64"
        return c
    lo, hi = {"blocks": (0.1, 1.0), "many": (0.001, 0.01), "mixed": (0.01, 0.2), "rmat": (0.004, 0.25),
              "grid": (0.02, 0.35)}[c["graph"]]
    if c["path"] == "plain":
        hi = {"mixed": 0.1, "grid": 0.25}.get(c["graph"], hi)
    c["scale"] = round(_log(rng, lo, hi), 5)
    if c["path"] == "batched":
        c["precision"] = rng.choice(["fp64", "fp32c"])
    if c["sources"]:
        c["pick"] = rng.choice(["random", "tiles"])
        c["sources"] = int(_log(rng, 64, c["sources"]))
        if c["pick"] == "random":
            c["sources"] = min(c["sources"], 2001)
    return c


# ------------------------------------------------------------------ inputs
def _edges(case, seed):
    """(n, uv) of the case's graph from the seed alone.  The generators fix
    the graph by workload and scale; the seed draws its vertex numbers and the
    order and direction of its edges, which decide the order that the
    decomposition finds blocks and local numbers in."""
    rng = np.random.default_rng(int(seed))
    if case["graph"] != "ring":
        n, uv = bcx.generate(WORKLOADS[case["graph"]], 0, float(case["scale"]))
        uv = rng.permutation(n).astype(np.int32)[uv[rng.permutation(len(uv))]]
        flip = rng.random(len(uv)) < 0.5
        uv[flip] = uv[flip][:, ::-1]
        return n, np.ascontiguousarray(uv)
    n = int(case["n"])
    order = rng.permutation(n)
    ring = np.stack([order, np.roll(order, -1)], 1)
    chords = max(1, int(n * (float(case["degree"]) - 2) / 2))
    uv = np.concatenate([ring, rng.integers(0, n, size=(chords, 2))])
    uv = uv[uv[:, 0] != uv[:, 1]]
    lo, hi = uv.min(1), uv.max(1)
    _, first = np.unique(lo.astype(np.int64) * n + hi, return_index=True)
    return n, np.ascontiguousarray(uv[rng.permutation(first)], dtype=np.int32)


def _reduced(case, seed):
    n, uv = _edges(case, seed)
    return bcx.Host.from_edges(n, uv).decompose(use_chains=case["chains"])


def _random_slots(case, seed, comps):
    """Slots of `sources` vertices of the largest component, or None for all."""
    sizes = np.array([c.n for c in comps], np.int64)
    big = int(sizes.argmax())
    k = min(int(case["sources"]), int(sizes[big]))
    rng = np.random.default_rng([int(seed), 77])
    return int(sizes[:big].sum()) + np.sort(rng.choice(int(sizes[big]), size=k, replace=False)).astype(np.int64)


def _tile_slots(case, comps, order, big):
    """Slots of `sources` vertices of component `big`: runs of 256 evenly
    spaced over the library's order of it."""
    n, k = len(order), min(int(case["sources"]), len(order))
    starts = np.linspace(0, max(0, n - 256), -(-k // 256)).astype(np.int64)
    at = np.unique(starts[:, None] + np.arange(256)[None, :])
    at = at[at < n][:k]
    return int(sum(c.n for c in comps[:big])) + np.sort(order[at].astype(np.int64))


_engine = None


def _get_engine():
    """The process's one engine, as a program keeps it."""
    global _engine
    if _engine is None:
        _engine = bcx.Engine(0)
    return _engine


class State:
    """What a program has in hand before the call; gives its device graph back."""
    graph = None

    def __del__(self):
        if self.graph is not None:
            self.graph.free()
            self.graph = None


def prepare(case, seed):
    s = State()
    s.entry = case["entry"]
    s.options = dict(path=PATHS[case["path"]], precision=PRECISIONS[case["precision"]], use_chains=case["chains"])
    s.engine = _get_engine()
    s.host = _reduced(case, seed)
    if s.entry == "host":
        return s
    comps = s.host.components()
    if s.entry == "device":
        c = comps[0]
        s.n, s.arcs = c.n, c.arcs
        s.inputs = [torch.from_numpy(np.ascontiguousarray(x, dtype=np.int32)).cuda()
                    for x in (c.row_ptr, c.col, c.reach)]
        s.bc = torch.zeros(c.n, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        return s
    s.graph = s.engine.upload(comps)
    if case["sources"] and case["pick"] == "tiles":
        big = max(range(len(comps)), key=lambda i: comps[i].n)
        s.options["subset"] = _tile_slots(case, comps, s.graph.batched_order(big), big)
    elif case["sources"]:
        s.options["subset"] = _random_slots(case, seed, comps)
    return s


def run(s):
    if s.entry == "host":
        return s.engine.host_bc(s.host, **s.options)[0]
    if s.entry == "run":
        return s.graph.run(**s.options)[0]
    # the call runs on the engine's own stream and adds to bc, which the
    # caller's stream has to have cleared by then
    s.bc.zero_()
    torch.cuda.current_stream().synchronize()
    ptr = [ctypes.c_void_p(t.data_ptr()) for t in (*s.inputs, s.bc)]
    rc = bcx.lib().bcx_bc_small_noalloc(s.engine.h, s.n, s.arcs, ptr[0], ptr[1], ptr[2], None, 0,
                                        s.options["precision"], ptr[3])
    if rc:
        raise bcx.BcxError(rc, bcx.lib().bcx_last_error(s.engine.h).decode())
    return s.bc


# -------------------------------------------------------------------- work
def _sizes(case):
    """(vertices, arcs, sum over sources of their component's arcs, sum over
    sources of its vertices) by the generators' nominal sizes."""
    if case["graph"] == "ring":
        n = case["n"]
        a = n * case["degree"]
        return n, a, n * a, n * n
    s = case["scale"]
    if case["graph"] == "blocks":
        k = max(2, round(16 * s))
        return 600 * k, 2050 * k, 600 * 2050 * k, 600 * 600 * k
    if case["graph"] == "many":
        # block sizes are log-uniform in 3..2000, arcs about 8 per vertex
        k, core, core_arcs = 40000 * s, 544e3 * s, 9e6 * s
        sq = (2000 ** 2 - 9) / (2 * math.log(2000 / 3))
        return 307 * k + core, 2457 * k + core_arcs, 8 * sq * k + core * core_arcs, sq * k + core * core
    n, a = {"mixed": (838e3, 12.6e6), "grid": (74.5e3, 266e3), "rmat": (660e3, 30.4e6)}[case["graph"]]
    n, a = n * s, a * s
    k = min(case["sources"] or n, n)
    return n, a, k * a, k * n


def work(case):
    n, arcs, src_arcs, src_n = _sizes(case)
    # graph, weights and result once; per source half the arcs (an edge lies
    # on shortest paths in one direction) add a path count and a dependency
    # term, and a vertex divides, adds, multiplies and accumulates
    return {"bytes": 4.0 * (n + 1) + 4.0 * arcs + 4.0 * n + 8.0 * n, "flops": 1.0 * src_arcs + 5.0 * src_n}


# ------------------------------------------------------------------- exact
def _weighted_brandes(rp, col, reach, comp, sources):
    """Sum over sources s of (reach[s] + 1) times the dependencies of s with
    target weights reach + 1, in 64 bits: level-synchronous Brandes over a
    block-diagonal graph.  comp[v] is the block of v; column k of the state
    holds the k-th source of every block at once."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    n = len(rp) - 1
    graph = torch.sparse_csr_tensor(torch.from_numpy(rp), torch.from_numpy(col), torch.ones(len(col), dtype=torch.float64),
                                    size=(n, n)).to(dev)
    weight = torch.from_numpy(reach.astype(np.float64) + 1.0).to(dev)
    block = torch.from_numpy(comp).to(dev)
    n_blocks = int(comp.max()) + 1
    # k-th source of its block
    ss = sources[np.argsort(comp[sources], kind="stable")]
    head = np.concatenate([[0], np.flatnonzero(np.diff(comp[ss])) + 1])
    k_of = np.arange(len(ss)) - np.repeat(head, np.diff(np.append(head, len(ss))))
    bc = torch.zeros(n, dtype=torch.float64, device=dev)
    for k0 in range(0, int(k_of.max()) + 1, 512):
        pick = (k_of >= k0) & (k_of < k0 + 512)
        s = torch.from_numpy(ss[pick]).to(dev)
        k = torch.from_numpy(k_of[pick] - k0).to(dev)
        w = int(k.max()) + 1
        wsrc = torch.zeros((n_blocks, w), dtype=torch.float64, device=dev)
        wsrc[block[s], k] = weight[s]
        level = torch.full((n, w), -1, dtype=torch.int32, device=dev)
        sigma = torch.ones((n, w), dtype=torch.float64, device=dev)
        level[s, k] = 0
        depth = 0
        front = torch.zeros((n, w), dtype=torch.float64, device=dev)  # sigma on the last level, else 0
        front[s, k] = 1.0
        while True:
            front = graph @ front
            new = (level < 0) & (front > 0)
            if not bool(new.any()):
                break
            depth += 1
            level[new] = depth
            front *= new
            torch.where(new, front, sigma, out=sigma)
        rho = torch.zeros_like(sigma)
        delta = torch.zeros_like(sigma)
        for l in range(depth, 0, -1):
            here = level == l
            delta = torch.where(here, sigma * rho, delta)
            rho = graph @ torch.where(here, (weight[:, None] + delta) / sigma, 0.0)
        bc += (delta * wsrc[block]).sum(1)
    return bc.cpu().numpy()


def exact(case, seed):
    _, arcs, src_arcs, _ = _sizes(case)
    if src_arcs > 8e10:
        return None
    host = _reduced(case, seed)
    comps = host.components()  # the inputs: blocks, reach weights
    if not comps:
        return np.asarray(host.cut_term(), np.float64)
    off = np.concatenate([[0], np.cumsum([c.n for c in comps])]).astype(np.int64)
    rp = np.concatenate([[0]] + [c.row_ptr[1:].astype(np.int64) for c in comps])
    base = np.concatenate([[0], np.cumsum([c.arcs for c in comps])])
    for i in range(len(comps)):
        rp[off[i] + 1:off[i + 1] + 1] += base[i]
    col = np.concatenate([c.col.astype(np.int64) + off[i] for i, c in enumerate(comps)])
    reach = np.concatenate([c.reach for c in comps])
    block = np.repeat(np.arange(len(comps), dtype=np.int64), np.diff(off))
    if case["sources"] and case["pick"] == "tiles":
        # the order that the tiles are cut from is an input
        g = _get_engine().upload(comps)
        big = max(range(len(comps)), key=lambda i: comps[i].n)
        sources = _tile_slots(case, comps, g.batched_order(big), big)
        g.free()
    elif case["sources"]:
        sources = _random_slots(case, seed, comps)
    else:
        sources = np.arange(off[-1], dtype=np.int64)
    bc = _weighted_brandes(rp, col, reach, block, sources)
    if case["entry"] != "host":
        return bc
    out = np.asarray(host.cut_term(), np.float64)  # pairs that a cut vertex separates
    for i, c in enumerate(comps):
        out[c.gid] += bc[off[i]:off[i + 1]]
    return out
