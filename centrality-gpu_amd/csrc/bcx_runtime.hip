// GPU engine half of the C-ABI (include/bcx.h): context, device memory with a
// hard cap, component upload, source planning (free sources, endpoint rows,
// chain batches) and the launch sequence of the plain and batched paths.
//
// Replaces the reference's begin_gpu / bc_gpu_free / bc_gpu_active /
// postprocess host drivers (Codes/begin_gpupgm.cu:42-89,
// Codes/kernels_free.cu:6-114, Codes/kernels_active.cu:18-223,
// Codes/postprocesses.cu:8-203): one upload of all components instead of a
// malloc/copy/free per BCC, status codes instead of exit().
#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "../host/host_graph.h"
#include "bcx.h"
#include "bcx_batched.h"
#include "bcx_device.h"
#include "bcx_kernels.h"
#include "bcx_src.h"
#include "bcx_runtime.h"
#include "bcx_small.h"

using namespace bcx;

// ------------------------------------------------------------------------
// context and memory
// ------------------------------------------------------------------------

int ctx_fail(bcx_ctx *ctx, int code, const std::string &msg) {
    if (ctx) ctx->err = msg;
    return code;
}

int ctx_hip(bcx_ctx *ctx, hipError_t e, const char *what) {
    if (e == hipSuccess) return BCX_OK;
    return ctx_fail(ctx, e == hipErrorOutOfMemory ? BCX_E_NOMEM : BCX_E_HIP,
                    std::string(what) + ": " + hipGetErrorString(e));
}

// The per-source kernel's rows and accumulators are kept from run to run for
// speed alone: where an allocation finds no room beside them they are given
// back (hipFree waits for what still runs on them).
static bool give_rows_back(bcx_ctx *ctx) {
    bool any = false;
    auto give = [&](DBuf &b) {
        any |= b.p != nullptr;
        b.release(ctx);
    };
    if (!ctx->rows_held) {
        give(ctx->plain_scratch);
        give(ctx->bc_split);
    }
    if (!ctx->copies_held) give(ctx->bc_copies);
    return any;
}

size_t ctx_room(const bcx_ctx *ctx) {
    const size_t rows = (ctx->rows_held ? 0 : ctx->plain_scratch.bytes + ctx->bc_split.bytes) +
                        (ctx->copies_held ? 0 : ctx->bc_copies.bytes);
    return ctx->mem_cap + rows > ctx->mem_used ? ctx->mem_cap + rows - ctx->mem_used : 0;
}

int dev_alloc(bcx_ctx *ctx, void **p, size_t bytes, const char *what) {
    *p = nullptr;
    if (bytes == 0) bytes = 64;
    bytes = (bytes + 255) & ~(size_t)255;
    if (ctx->mem_used + bytes > ctx->mem_cap && ctx_room(ctx) >= bytes) (void)give_rows_back(ctx);
    if (ctx->mem_used + bytes > ctx->mem_cap)
        return ctx_fail(ctx, BCX_E_NOMEM,
                        std::string("device memory cap exceeded allocating ") + what + " (" +
                            std::to_string(bytes) + " B, " + std::to_string(ctx->mem_used) +
                            " of " + std::to_string(ctx->mem_cap) + " B in use)");
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory && give_rows_back(ctx)) {
        (void)hipGetLastError();
        e = hipMalloc(p, bytes);
    }
    if (e != hipSuccess) {
        *p = nullptr;
        return ctx_hip(ctx, e, what);
    }
    ctx->mem_used += bytes;
    ctx->sizes[*p] = bytes;
    return BCX_OK;
}

void dev_free(bcx_ctx *ctx, void *p) {
    if (!p) return;
    auto it = ctx->sizes.find(p);
    if (it != ctx->sizes.end()) {
        ctx->mem_used -= it->second;
        ctx->sizes.erase(it);
    }
    (void)hipFree(p);
}

int DBuf::ensure(bcx_ctx *ctx, size_t need, const char *what) {
    if (need <= bytes && p) return BCX_OK;
    dev_free(ctx, p);
    p = nullptr;
    bytes = 0;
    size_t grow = need + need / 8;
    int rc = dev_alloc(ctx, &p, grow, what);
    if (rc) {
        rc = dev_alloc(ctx, &p, need, what);
        if (rc) return rc;
        bytes = need;
        return BCX_OK;
    }
    bytes = grow;
    return BCX_OK;
}

void DBuf::release(bcx_ctx *ctx) {
    dev_free(ctx, p);
    p = nullptr;
    bytes = 0;
}

int upload(bcx_ctx *ctx, const void *host, size_t bytes, DBuf &buf, const char *what) {
    int rc = buf.ensure(ctx, bytes ? bytes : 4, what);
    if (rc) return rc;
    if (bytes) return ctx_hip(ctx, hipMemcpyAsync(buf.p, host, bytes, hipMemcpyHostToDevice, ctx->stream), what);
    return BCX_OK;
}

// Kernel time: events around every launch, summed after the final sync.
void Timer::begin(bcx_ctx *ctx) {
    if (depth++ > 0) return;
    if (used == evs.size()) {
        hipEvent_t a, b;
        (void)hipEventCreate(&a);
        (void)hipEventCreate(&b);
        evs.push_back({a, b});
    }
    (void)hipEventRecord(evs[used].first, ctx->stream);
}
void Timer::end(bcx_ctx *ctx) {
    if (--depth > 0) return;
    (void)hipEventRecord(evs[used].second, ctx->stream);
    used++;
}
double Timer::collect() {
    double t = 0;
    for (size_t i = 0; i < used; ++i) {
        float ms = 0;
        (void)hipEventSynchronize(evs[i].second);
        (void)hipEventElapsedTime(&ms, evs[i].first, evs[i].second);
        t += ms * 1e-3;
    }
    used = 0;
    return t;
}
void Timer::destroy() {
    for (auto &e : evs) {
        (void)hipEventDestroy(e.first);
        (void)hipEventDestroy(e.second);
    }
    evs.clear();
    used = 0;
}

// ------------------------------------------------------------------------
// source planning
// ------------------------------------------------------------------------

// Roles, chain membership and the chain batches for one component.
// Every endpoint of a needed chain gets its own BC exactly once (MODE_BC)
// in the first batch that holds its row; later batches recompute the row
// only (MODE_ROW).  Chains are ordered by the BFS position of their later
// endpoint on the ear graph (endpoints as vertices, chains as edges), the
// role of the ear-graph level batches of Codes/arrangelevels.cpp:56-109, and
// packed greedily while the distinct endpoints fit in row_cap slots.
// With `direct`, the sources of a chain whose endpoints' rows only it needs run
// as BFS sources: on an 84k power-law core a kept row costs 10.2 us, a combined
// source 9.5 us and a BFS source 13.4 us, so a row that no source wants for
// itself pays from three chain sources on; and the combine's launches of their
// own pay from an eighth of the sources on (1000 sampled sources 18.9 -> 13.5
// ms, 2049 of an 18.6k grid 5.1 -> 3.5 ms; with every source of a 17k core
// wanted, 37% of them on chains, the rows save 6%).
int bcx::make_plan(const HostComp &hc, const int32_t *subset, int64_t n_sub, bool use_chains,
              int64_t row_cap, bool direct, Plan &plan) {
    const int32_t n = hc.n;
    const int32_t nch = use_chains ? hc.n_chains : 0;
    plan = Plan();
    std::vector<int32_t> chain_of((size_t)n, -1), pos_of((size_t)n, -1);
    std::vector<uint8_t> is_end((size_t)n, 0);
    for (int32_t c = 0; c < nch; ++c) {
        for (int32_t j = hc.ch_ptr[c]; j < hc.ch_ptr[c + 1]; ++j) {
            chain_of[hc.ch_nodes[j]] = c;
            pos_of[hc.ch_nodes[j]] = j - hc.ch_ptr[c];
        }
        is_end[hc.ch_ends[2 * c]] = 1;
        is_end[hc.ch_ends[2 * c + 1]] = 1;
    }
    std::vector<uint8_t> want_bfs((size_t)n, 0);
    std::vector<std::vector<int32_t>> chain_srcs((size_t)nch);
    int64_t n_wanted = 0;
    auto add = [&](int32_t v) {
        if (v < 0 || v >= n) return;
        n_wanted++;
        if (chain_of[v] >= 0) chain_srcs[chain_of[v]].push_back(pos_of[v]);
        else want_bfs[v] = 1;
    };
    if (subset) for (int64_t i = 0; i < n_sub; ++i) add(subset[i]);
    else for (int32_t v = 0; v < n; ++v) add(v);

    std::vector<int32_t> need;  // needed chains
    for (int32_t c = 0; c < nch; ++c)
        if (!chain_srcs[c].empty()) {
            std::sort(chain_srcs[c].begin(), chain_srcs[c].end());
            chain_srcs[c].erase(std::unique(chain_srcs[c].begin(), chain_srcs[c].end()), chain_srcs[c].end());
            need.push_back(c);
        }
    if (direct) {
        auto pays = [&](int32_t c) {
            const int32_t L = hc.ch_ends[2 * c], R = hc.ch_ends[2 * c + 1];
            const size_t rows = (size_t)!want_bfs[L] + (size_t)(!want_bfs[R] && R != L);
            return chain_srcs[c].size() >= 3 * rows;
        };
        int64_t combined = 0;
        for (int32_t c : need)
            if (pays(c)) combined += (int64_t)chain_srcs[c].size();
        const bool none = combined < n_wanted / 8;
        std::vector<int32_t> keep;
        for (int32_t c : need) {
            if (!none && pays(c)) {
                keep.push_back(c);
                continue;
            }
            for (int32_t p : chain_srcs[c]) plan.free_src.push_back(hc.ch_nodes[hc.ch_ptr[c] + p]);
            plan.n_chain += (int64_t)chain_srcs[c].size();
        }
        need.swap(keep);
    }
    const int64_t n_direct = (int64_t)plan.free_src.size();
    // endpoints of needed chains
    std::vector<uint8_t> needed_end((size_t)n, 0);
    for (int32_t c : need) {
        needed_end[hc.ch_ends[2 * c]] = 1;
        needed_end[hc.ch_ends[2 * c + 1]] = 1;
    }
    for (int32_t v = 0; v < n; ++v)
        if (want_bfs[v] && !needed_end[v]) plan.free_src.push_back(v);
    plan.n_bfs = (int64_t)plan.free_src.size() - n_direct;
    if (need.empty()) return BCX_OK;

    // ear graph BFS order over needed endpoints
    std::vector<std::vector<int32_t>> eadj;
    std::vector<int32_t> eid((size_t)n, -1), everts;
    for (int32_t c : need)
        for (int k = 0; k < 2; ++k) {
            int32_t v = hc.ch_ends[2 * c + k];
            if (eid[v] < 0) { eid[v] = (int32_t)everts.size(); everts.push_back(v); }
        }
    eadj.assign(everts.size(), {});
    for (int32_t c : need) {
        int32_t a = eid[hc.ch_ends[2 * c]], b = eid[hc.ch_ends[2 * c + 1]];
        eadj[a].push_back(b);
        eadj[b].push_back(a);
    }
    std::vector<int32_t> bpos(everts.size(), -1);
    int32_t cntpos = 0;
    std::vector<int32_t> q;
    for (size_t r = 0; r < everts.size(); ++r) {
        if (bpos[r] >= 0) continue;
        q.clear();
        q.push_back((int32_t)r);
        bpos[r] = cntpos++;
        for (size_t i = 0; i < q.size(); ++i)
            for (int32_t y : eadj[q[i]])
                if (bpos[y] < 0) { bpos[y] = cntpos++; q.push_back(y); }
    }
    std::vector<std::pair<int64_t, int32_t>> order;
    for (int32_t c : need) {
        int32_t a = bpos[eid[hc.ch_ends[2 * c]]], b = bpos[eid[hc.ch_ends[2 * c + 1]]];
        order.push_back({(int64_t)std::max(a, b) * (1ll << 31) + std::min(a, b), c});
    }
    std::sort(order.begin(), order.end());

    if (row_cap < 2) row_cap = 2;
    std::vector<uint8_t> bc_done((size_t)n, 0);
    std::vector<int32_t> slot((size_t)n, -1);
    PlanBatch cur;
    std::vector<int32_t> cur_ends;
    auto flush = [&]() {
        if (cur_ends.empty()) return;
        for (int32_t v : cur_ends) {
            int8_t mode = MODE_ROW;
            if (want_bfs[v] && !bc_done[v]) { mode |= MODE_BC; bc_done[v] = 1; plan.n_bfs++; }
            else plan.n_row_only++;
            cur.bsrc.push_back(v);
            cur.bslot.push_back(slot[v]);
            cur.bmode.push_back(mode);
        }
        for (int32_t v : cur_ends) slot[v] = -1;
        cur.n_rows = (int32_t)cur_ends.size();
        plan.batches.push_back(std::move(cur));
        cur = PlanBatch();
        cur_ends.clear();
    };
    for (auto &pr : order) {
        int32_t c = pr.second;
        int32_t L = hc.ch_ends[2 * c], R = hc.ch_ends[2 * c + 1];
        int extra = (slot[L] < 0) + (slot[R] < 0 && R != L);
        if ((int64_t)cur_ends.size() + extra > row_cap) flush();
        for (int32_t v : {L, R})
            if (slot[v] < 0) { slot[v] = (int32_t)cur_ends.size(); cur_ends.push_back(v); }
        for (int32_t p : chain_srcs[c]) {
            cur.cci.push_back(c);
            cur.cpos.push_back(p);
            cur.cslots.push_back(slot[L]);
            cur.cslots.push_back(slot[R]);
            plan.n_chain++;
        }
    }
    flush();
    // endpoints that wanted BC but were never placed (cannot happen: every
    // needed endpoint is in some batch) -- keep the invariant explicit
    for (int32_t v : everts)
        if (want_bfs[v] && !bc_done[v]) { plan.free_src.push_back(v); plan.n_bfs++; }
    return BCX_OK;
}

// ------------------------------------------------------------------------
// plain path
// ------------------------------------------------------------------------

static int64_t plain_stride(int32_t n) { return ((int64_t)n + 2 + 63) & ~(int64_t)63; }
constexpr size_t PLAIN_WORD_BYTES = 4 + 8 + 8 + 4 + 4;  // d, sig, dl, S, off

// Device memory for the workgroups' rows: what they hold now plus what the cap leaves.
static size_t plain_room(bcx_ctx *ctx) {
    const size_t others = ctx->mem_used - ctx->plain_scratch.bytes;
    return std::max(ctx->plain_scratch.bytes, ctx->mem_cap > others ? ctx->mem_cap - others : 0);
}

// Fewest workgroups a run of `count` sources takes: with less memory than
// their rows it is refused.
static int64_t plain_min_grid(bcx_ctx *ctx, int64_t count) {
    return std::max<int64_t>(1, std::min<int64_t>(count, 2 * (int64_t)ctx->n_cu));
}

bool plain_scratch_fits(bcx_ctx *ctx, int32_t n, int64_t count) {
    return (size_t)plain_stride(n) * PLAIN_WORD_BYTES * (size_t)plain_min_grid(ctx, count) <= plain_room(ctx);
}

// Workgroups of a launch: what the compute units hold, within the sources and
// half of the device memory that is left.
static int plain_grid(bcx_ctx *ctx, int32_t n, int64_t count, const PlainShape &p) {
    const int64_t fit = (int64_t)(plain_room(ctx) / 2 / ((size_t)plain_stride(n) * PLAIN_WORD_BYTES));
    const int64_t g = std::min<int64_t>({count, (int64_t)ctx->n_cu * p.per_cu, fit});
    return (int)std::max(g, plain_min_grid(ctx, count));
}

// While it lives, the context's rows belong to a launch being put together.
struct RowsHeld {
    bcx_ctx *ctx;
    explicit RowsHeld(bcx_ctx *c) : ctx(c) { ctx->rows_held++; }
    ~RowsHeld() { ctx->rows_held--; }
};

static int ensure_plain_scratch(bcx_ctx *ctx, int32_t n, int grid, PlainScratch &sc) {
    const int64_t stride = plain_stride(n);
    const size_t per = (size_t)stride * PLAIN_WORD_BYTES;
    int rc = ctx->plain_scratch.ensure(ctx, per * (size_t)grid, "plain scratch");
    if (rc) return rc;
    char *p = (char *)ctx->plain_scratch.p;
    const size_t g = (size_t)grid * stride;
    sc.stride = stride;
    sc.sig = (uint64_t *)p; p += g * 8;
    sc.dl = (double *)p;    p += g * 8;
    sc.d = (int32_t *)p;    p += g * 4;
    sc.S = (int32_t *)p;    p += g * 4;
    sc.off = (int32_t *)p;
    return BCX_OK;
}

static int ensure_rows(bcx_ctx *ctx, int32_t n, int32_t nrows, Rows &rows) {
    const int64_t stride = ((int64_t)n + 63) & ~(int64_t)63;
    const size_t bytes = (size_t)stride * 12 * (size_t)std::max(nrows, 1);
    int rc = ctx->rows_buf.ensure(ctx, bytes, "endpoint rows");
    if (rc) return rc;
    rows.stride = stride;
    rows.sig = (uint64_t *)ctx->rows_buf.p;
    rows.d = (int32_t *)((char *)ctx->rows_buf.p + (size_t)stride * 8 * std::max(nrows, 1));
    return BCX_OK;
}

int64_t row_capacity(bcx_ctx *ctx, int32_t n, const bcx_opts *o) {
    const int64_t per = (((int64_t)n + 63) & ~(int64_t)63) * 12;
    int64_t cap = (o && o->row_cap_bytes > 0) ? o->row_cap_bytes : (int64_t)(ctx->mem_cap / 4);
    int64_t r = cap / std::max<int64_t>(per, 1);
    return std::max<int64_t>(2, std::min<int64_t>(r, 1 << 16));
}

// (ordered: on the ordered copy when there is one; no rows kept)
static int run_bfs_list(bcx_ctx *ctx, const DComp &dc, const std::vector<int32_t> &src,
                        const std::vector<int32_t> &slot, const std::vector<int8_t> &mode,
                        bool f64, uint64_t limit, double *bc, const Rows &rows, bcx_stats *st,
                        double *probe = nullptr, bool fp32 = false, bool ordered = false) {
    if (src.empty()) return BCX_OK;
    int rc;
    const RowsHeld held(ctx);
    if ((rc = ctx->w_src.ensure(ctx, src.size() * 4, "work list"))) return rc;
    if ((rc = upload(ctx, slot.data(), slot.size() * 4, ctx->w_aux, "work list"))) return rc;
    if ((rc = upload(ctx, mode.data(), mode.size(), ctx->w_mode, "work list"))) return rc;
    rc = ctx_hip(ctx, hipMemsetAsync(ctx->counters.p, 0, 4 * sizeof(int32_t), ctx->stream), "memset");
    if (rc) return rc;
    const PlainShape shape = plain_shape(dc.n, fp32);
    const int grid = plain_grid(ctx, dc.n, (int64_t)src.size(), shape);
    PlainScratch sc;
    if ((rc = ensure_plain_scratch(ctx, dc.n, grid, sc))) return rc;
    // The sources add into copies of the accumulator, one per eight of them up to
    // SPLIT, folded afterwards: a vertex's sum is then that much shorter, and its
    // rounding error what the tiled kernels' is, which add a tile's sources in pairs
    // (error in the sum alone on a grid of 3600 vertices, FP64 terms, with one
    // accumulator / so: 64 sources 1.3 / 0.44 ulp, 361 sources 3.1 / 0.44, 1500
    // sources - / 0.56; 32 copies 0.33 and 0.41 for the latter two, but 2049 sources
    // of an 18.6k grid 3.20 -> 3.25 ms).  With FP32 terms the terms' own rounding
    // hides it, and only hundreds of sources and more take copies.  Accumulators of
    // the workgroups' own, without atomics, ran 20-30% slower (8000 sources of a 26k
    // grid 13.6 -> 16.0 ms).  Where a capacity has little room left beside the rows
    // above, there are fewer, and without room for one an ordered run has the
    // component's own order.
    constexpr int SPLIT = 16;
    constexpr size_t SPLIT_FP32 = 512;
    const size_t word = sizeof(double) * (size_t)dc.n;
    const size_t room = ctx->mem_cap > ctx->mem_used ? ctx->mem_cap - ctx->mem_used : 0;
    int split = fp32 && src.size() < SPLIT_FP32 ? 1 : SPLIT;
    while (split > 1 && (8 * (size_t)split > src.size() || ctx->bc_split.bytes + room / 16 < word * split)) split /= 2;
    ordered = ordered && dc.ord_state == 1;
    if (split > 1 && ctx->bc_split.ensure(ctx, word * split, "split accumulator") != BCX_OK) split = 1;
    if (ordered && split == 1 && ctx->bc_split.ensure(ctx, word, "accumulator") != BCX_OK) ordered = false;
    const bool fold = split > 1 || ordered;  // (an ordered run folds its one copy back to the component's order)
    std::vector<int32_t> ids;
    if (ordered)
        for (int32_t v : src) ids.push_back(dc.ord_inv[(size_t)v]);
    if ((rc = upload(ctx, ordered ? ids.data() : src.data(), src.size() * 4, ctx->w_src, "work list"))) return rc;
    PlainArgs a{};
    a.src = (const int32_t *)ctx->w_src.p;
    a.aux = (const int32_t *)ctx->w_aux.p;
    a.mode = (const int8_t *)ctx->w_mode.p;
    a.count = (int32_t)src.size();
    a.sigma_f64 = f64;
    a.limit = limit;
    a.counters = (int32_t *)ctx->counters.p;
    a.bc = bc;
    a.probe = probe;
    a.fp32 = fp32;
    a.sweep = plain_sweep(dc.n, dc.arcs);
    a.split = split;
    if (fold) {
        a.bc = (double *)ctx->bc_split.p;
        if ((rc = ctx_hip(ctx, hipMemsetAsync(a.bc, 0, word * a.split, ctx->stream), "memset"))) return rc;
    }
    ctx->timer.begin(ctx);
    hipError_t e = launch_plain_bfs(ordered ? dc.ord : dc.dev, a, sc, rows, shape, grid, ctx->stream);
    if (e == hipSuccess && fold)
        e = launch_plain_fold(bc, a.bc, ordered ? dc.ord_perm : nullptr, dc.n, a.split, ctx->stream);
    ctx->timer.end(ctx);
    if (st) st->n_launches += fold ? 2 : 1;
    rc = ctx_hip(ctx, e, "k_plain_bfs launch");
    if (rc) return rc;
    return read_counters(ctx, st);
}

// A copy of the component numbered in BFS order from its highest-degree vertex,
// for the per-source kernel: most gathers of a skewed graph go to few vertices,
// and those and what a level reaches then share cache lines (1000 sources of an
// 84k power-law core 13.5 -> 11.0 ms; ordered by degree class 12.4).  Rows keep
// the order of their arcs, so FP64 counts keep the oracle's sums.  Made for
// runs of ORDER_SOURCES sources or more, on components of ORDER_N vertices or
// more a quarter of whose vertices take half of the arcs (on grids the
// component's own order is as good).  The order is the vertex list that the
// kernel itself leaves behind for that source.
constexpr int32_t ORDER_N = 4096;
constexpr int64_t ORDER_SOURCES = 512;
static int order_copy(bcx_ctx *ctx, DComp &dc) {
    if (dc.ord_state >= 0) return BCX_OK;
    dc.ord_state = 0;
    const HostComp &h = dc.host;
    const int32_t n = h.n;
    if (n < ORDER_N) return BCX_OK;
    int64_t of[33] = {0}, arcs[33] = {0};  // vertices and arcs by degree class (powers of two)
    int32_t root = 0;
    for (int32_t v = 0; v < n; ++v) {
        const int32_t d = h.rp[v + 1] - h.rp[v];
        const int k = d > 0 ? 32 - __builtin_clz((unsigned)d) : 0;
        of[k]++;
        arcs[k] += d;
        if (d > h.rp[root + 1] - h.rp[root]) root = v;
    }
    int64_t top = 0, top_arcs = 0;
    for (int k = 32; k >= 0 && top + of[k] <= n / 4; --k) {
        top += of[k];
        top_arcs += arcs[k];
    }
    if (2 * top_arcs < h.arcs) return BCX_OK;
    // (a capacity that has little left beside the rows of a run goes without)
    const size_t copy = 4 * (4 * (size_t)n + 1 + h.col.size());
    const size_t rows = (size_t)plain_stride(n) * PLAIN_WORD_BYTES * (size_t)plain_min_grid(ctx, n);
    if (plain_room(ctx) < copy + rows + ctx->mem_cap / 4) return BCX_OK;
    int rc = run_bfs_list(ctx, dc, {root}, {-1}, {0}, true, 0, nullptr, Rows{}, nullptr);  // (forward only)
    PlainScratch sc;
    if (rc || (rc = ensure_plain_scratch(ctx, n, 1, sc))) return rc;
    // row pointers, permutation and its inverse from the host; columns and
    // reach weights are filled in on the device
    std::vector<int32_t> t(3 * (size_t)n + 1);
    int32_t *rp = t.data(), *perm = rp + n + 1, *inv = perm + n;
    if ((rc = ctx_hip(ctx, hipMemcpyAsync(perm, sc.S, 4 * (size_t)n, hipMemcpyDeviceToHost, ctx->stream), "copy")) ||
        (rc = ctx_hip(ctx, hipStreamSynchronize(ctx->stream), "copy")))
        return rc;
    std::fill(inv, inv + n, -1);
    rp[0] = 0;
    for (int32_t i = 0; i < n; ++i) {
        const int32_t v = perm[i];
        if (v < 0 || v >= n || inv[v] >= 0) return BCX_OK;  // (not connected: the list is short)
        inv[v] = i;
        rp[i + 1] = rp[i] + (h.rp[v + 1] - h.rp[v]);
    }
    // (no room under the cap: the component's own order does as well)
    if (dc.b_ord.ensure(ctx, 4 * (t.size() + (size_t)n + h.col.size()), "ordered component") != BCX_OK) return BCX_OK;
    int32_t *d = (int32_t *)dc.b_ord.p;
    dc.ord.n = n;
    dc.ord.arcs = dc.arcs;
    dc.ord.rp = d;
    dc.ord_perm = d + n + 1;
    dc.ord.reach = d + t.size();
    dc.ord.col = dc.ord.reach + n;
    dc.ord_inv.assign(inv, inv + n);
    rc = upload(ctx, t.data(), 4 * t.size(), dc.b_ord, "ordered component");
    if (!rc) rc = ctx_hip(ctx, launch_plain_reorder(dc.dev, dc.ord, dc.ord_perm, dc.ord_perm + n, ctx->stream), "reorder");
    if (!rc) rc = ctx_hip(ctx, hipStreamSynchronize(ctx->stream), "ordered component");
    if (!rc) dc.ord_state = 1;
    return rc;
}

int read_counters(bcx_ctx *ctx, bcx_stats *st) {
    int32_t h[4];
    int rc = ctx_hip(ctx, hipMemcpyAsync(h, ctx->counters.p, sizeof(h), hipMemcpyDeviceToHost, ctx->stream),
                     "counters");
    if (rc) return rc;
    rc = ctx_hip(ctx, hipStreamSynchronize(ctx->stream), "kernel execution");
    if (rc) return rc;
    ctx->overflow |= h[1] != 0;
    if (st && h[2] > st->max_level) st->max_level = h[2];
    return BCX_OK;
}

static int run_chain_list(bcx_ctx *ctx, const DComp &dc, const PlanBatch &b, bool f64, double *bc,
                          const Rows &rows, bcx_stats *st, double *probe = nullptr) {
    if (b.cci.empty()) return BCX_OK;
    int rc;
    const RowsHeld held(ctx);
    if ((rc = upload(ctx, b.cci.data(), b.cci.size() * 4, ctx->w_src, "chain list"))) return rc;
    if ((rc = upload(ctx, b.cpos.data(), b.cpos.size() * 4, ctx->w_aux, "chain list"))) return rc;
    if ((rc = upload(ctx, b.cslots.data(), b.cslots.size() * 4, ctx->w_slots, "chain list"))) return rc;
    rc = ctx_hip(ctx, hipMemsetAsync(ctx->counters.p, 0, 4 * sizeof(int32_t), ctx->stream), "memset");
    if (rc) return rc;
    const PlainShape shape = plain_shape(dc.n, false);
    const int grid = plain_grid(ctx, dc.n, (int64_t)b.cci.size(), shape);
    PlainScratch sc;
    if ((rc = ensure_plain_scratch(ctx, dc.n, grid, sc))) return rc;
    PlainArgs a{};
    a.src = (const int32_t *)ctx->w_src.p;
    a.aux = (const int32_t *)ctx->w_aux.p;
    a.slots = (const int32_t *)ctx->w_slots.p;
    a.count = (int32_t)b.cci.size();
    a.sigma_f64 = f64;
    a.counters = (int32_t *)ctx->counters.p;
    a.bc = bc;
    a.probe = probe;
    ctx->timer_chain.begin(ctx);
    hipError_t e = launch_plain_chain(dc.dev, dc.chains, a, sc, rows, shape, grid, ctx->stream);
    ctx->timer_chain.end(ctx);
    if (st) st->n_launches++;
    rc = ctx_hip(ctx, e, "k_plain_chain launch");
    if (rc) return rc;
    return read_counters(ctx, st);
}

// One component on the plain path in one sigma mode.
static int plain_component_mode(bcx_ctx *ctx, const DComp &dc, const Plan &plan, bool f64,
                                uint64_t limit, double *bc, bcx_stats *st) {
    int rc;
    Rows rows{};
    int32_t max_rows = 1;
    for (auto &b : plan.batches) max_rows = std::max(max_rows, b.n_rows);
    if ((rc = ensure_rows(ctx, dc.n, max_rows, rows))) return rc;
    std::vector<int32_t> slots(plan.free_src.size(), -1);
    std::vector<int8_t> modes(plan.free_src.size(), MODE_BC);
    if ((rc = run_bfs_list(ctx, dc, plan.free_src, slots, modes, f64, limit, bc, rows, st, nullptr, false, true)))
        return rc;
    if (ctx->overflow && !f64) return BCX_OK;
    for (auto &b : plan.batches) {
        if ((rc = run_bfs_list(ctx, dc, b.bsrc, b.bslot, b.bmode, f64, limit, bc, rows, st))) return rc;
        if (ctx->overflow && !f64) return BCX_OK;
        if ((rc = run_chain_list(ctx, dc, b, f64, bc, rows, st))) return rc;
    }
    return BCX_OK;
}

int plain_component(bcx_ctx *ctx, DComp &dc, const Plan &plan, const bcx_opts *o,
                    double *bc, bcx_stats *st) {
    const uint64_t limit = (o && o->sigma_f64_threshold_log2 > 0 && o->sigma_f64_threshold_log2 < 64)
                               ? (1ull << o->sigma_f64_threshold_log2) : 0;
    ctx->overflow = false;
    int rc = (int64_t)plan.free_src.size() >= ORDER_SOURCES ? order_copy(ctx, dc) : BCX_OK;
    if (rc) return rc;
    rc = plain_component_mode(ctx, dc, plan, false, limit, bc, st);
    if (rc) return rc;
    if (!ctx->overflow) return BCX_OK;
    // sigma left uint64: redo the component with FP64 sigma (pull order)
    rc = ctx_hip(ctx, hipMemsetAsync(bc, 0, sizeof(double) * dc.n, ctx->stream), "memset");
    if (rc) return rc;
    if (st) st->n_f64_sigma += plan.n_bfs + plan.n_chain;
    ctx->overflow = false;
    return plain_component_mode(ctx, dc, plan, true, 0, bc, st);
}

int source_component(bcx_ctx *ctx, DComp &dc, const std::vector<int32_t> &srcs, const bcx_opts *o, double *bc,
                     bcx_stats *st, bool *overflow) {
    const uint64_t limit = (o->sigma_f64_threshold_log2 > 0 && o->sigma_f64_threshold_log2 < 64)
                               ? (1ull << o->sigma_f64_threshold_log2) : 0;
    const bool fp32 = o->precision == BCX_PREC_FP32C;
    const std::vector<int32_t> slots(srcs.size(), -1);
    const std::vector<int8_t> modes(srcs.size(), MODE_BC);
    const Rows rows{};
    *overflow = false;
    int rc;
    if ((int64_t)srcs.size() >= ORDER_SOURCES && (rc = order_copy(ctx, dc))) return rc;
    // components whose counts from their highest-degree vertex pass 2^62 start
    // with FP64 counts, as on the workgroup kernel
    if (dc.sigma_est <= 4.6e18) {
        ctx->overflow = false;
        if ((rc = run_bfs_list(ctx, dc, srcs, slots, modes, false, limit, bc, rows, st, nullptr, fp32, true)))
            return rc;
        if (!ctx->overflow) return BCX_OK;
        rc = ctx_hip(ctx, hipMemsetAsync(bc, 0, sizeof(double) * (size_t)dc.n, ctx->stream), "memset");
        if (rc || fp32) {
            if (!limit) dc.src_wrapped = true;
            *overflow = true;
            return rc;
        }
    }
    if (st) st->n_f64_sigma += (int64_t)srcs.size();
    return run_bfs_list(ctx, dc, srcs, slots, modes, true, 0, bc, rows, st, nullptr, false, true);
}

// ------------------------------------------------------------------------
// C-ABI
// ------------------------------------------------------------------------
extern "C" {

int bcx_create(bcx_ctx **out, int device, size_t mem_cap) {
    if (!out) return BCX_E_ARG;
    *out = nullptr;
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= 0) return BCX_E_NODEV;
    if (device < 0 || device >= count) return BCX_E_ARG;
    if (hipSetDevice(device) != hipSuccess) return BCX_E_HIP;
    bcx_ctx *ctx = new bcx_ctx();
    ctx->device = device;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess) { delete ctx; return BCX_E_HIP; }
    ctx->n_cu = prop.multiProcessorCount;
    ctx->name = prop.gcnArchName;
    size_t free_b = 0, total_b = 0;
    (void)hipMemGetInfo(&free_b, &total_b);
    ctx->mem_cap = mem_cap ? mem_cap : (size_t)(0.9 * (double)free_b);
    // a failed lookup is recorded there and reported by bcx_bc_small_noalloc;
    // every other entry point works without the array
    (void)noalloc_init(device);
    if (hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking) != hipSuccess) {
        delete ctx;
        return BCX_E_HIP;
    }
    if (ctx->counters.ensure(ctx, 64, "counters") != BCX_OK) {
        (void)hipStreamDestroy(ctx->stream);
        delete ctx;
        return BCX_E_NOMEM;
    }
    *out = ctx;
    return BCX_OK;
}

void bcx_destroy(bcx_ctx *ctx) {
    if (!ctx) return;
    (void)hipSetDevice(ctx->device);
    (void)hipStreamSynchronize(ctx->stream);
    for (DBuf *b : ctx->all_bufs()) b->release(ctx);
    batched_release(ctx);
    small_release(ctx);
    ctx->timer.destroy();
    ctx->timer_chain.destroy();
    if (ctx->bc_pin) (void)hipHostFree(ctx->bc_pin);
    if (ctx->up_pin) (void)hipHostFree(ctx->up_pin);
    if (ctx->side) (void)hipStreamDestroy(ctx->side);
    (void)hipStreamDestroy(ctx->stream);
    delete ctx;
}

const char *bcx_last_error(const bcx_ctx *ctx) { return ctx ? ctx->err.c_str() : "null context"; }

int bcx_device_info(bcx_ctx *ctx, int32_t *n_cu, char *name, int32_t name_len) {
    if (!ctx) return BCX_E_ARG;
    if (n_cu) *n_cu = ctx->n_cu;
    if (name && name_len > 0) {
        std::strncpy(name, ctx->name.c_str(), (size_t)name_len - 1);
        name[name_len - 1] = '\0';
    }
    return BCX_OK;
}

int bcx_upload(bcx_ctx *ctx, const bcx_component *comps, int32_t n_comps, bcx_dgraph **out) {
    if (!ctx || !out || n_comps < 0 || (n_comps > 0 && !comps)) return ctx_fail(ctx, BCX_E_ARG, "bad upload args");
    *out = nullptr;
    (void)hipSetDevice(ctx->device);
    bcx_dgraph *g = new bcx_dgraph();
    int64_t off = 0;
    for (int32_t i = 0; i < n_comps; ++i) {
        const bcx_component &c = comps[i];
        if (c.n <= 0 || !c.row_ptr || !c.col || !c.reach || c.row_ptr[0] != 0 || c.arcs != (int64_t)c.row_ptr[c.n] ||
            c.arcs >= INT32_MAX || (c.n_chains > 0 && (!c.chain_ptr || !c.chain_nodes || !c.chain_ends))) {
            bcx_dgraph_free(ctx, g);
            return ctx_fail(ctx, BCX_E_ARG, "component " + std::to_string(i) + " is malformed");
        }
        g->comps.emplace_back();
        DComp &dc = g->comps.back();
        HostComp &hc = dc.host;
        dc.n = c.n;
        dc.arcs = c.arcs;
        dc.offset = off;
        off += c.n;
        hc.n = c.n;
        hc.arcs = c.arcs;
        hc.rp.assign(c.row_ptr, c.row_ptr + c.n + 1);
        for (int32_t v = 0; v < c.n; ++v) dc.groups += (hc.rp[v + 1] - hc.rp[v] + 3) / 4;
        hc.col.assign(c.col, c.col + c.arcs);
        hc.reach.assign(c.reach, c.reach + c.n);
        hc.n_chains = std::max(c.n_chains, 0);
        if (hc.n_chains) {
            hc.ch_ptr.assign(c.chain_ptr, c.chain_ptr + c.n_chains + 1);
            hc.ch_nodes.assign(c.chain_nodes, c.chain_nodes + c.chain_ptr[c.n_chains]);
            hc.ch_ends.assign(c.chain_ends, c.chain_ends + 2 * c.n_chains);
        } else {
            hc.ch_ptr.assign(1, 0);
        }
    }
    g->total_n = off;
    for (const DComp &dc : g->comps) g->offs.push_back(dc.offset);
    // every array of every component in one device allocation and one copy
    // (tens of thousands of small components would otherwise cost an
    // allocation and a copy per array); arrays start on 256-byte boundaries
    auto padded = [](size_t k) { return (k + 63) & ~(size_t)63; };
    size_t words = 0;
    for (DComp &dc : g->comps) {
        const HostComp &hc = dc.host;
        words += padded(hc.rp.size()) + padded(hc.col.size()) + padded(hc.reach.size()) + padded(hc.ch_ptr.size()) +
                 padded(hc.ch_nodes.size()) + padded(hc.ch_ends.size());
    }
    int rc = g->pool.ensure(ctx, 4 * std::max<size_t>(words, 1), "components");
    if (rc) { bcx_dgraph_free(ctx, g); return rc; }
    // small sets go through a pinned buffer of the context and the copy is not
    // waited for: everything that reads them is ordered behind it.  Larger sets
    // are faster through a pageable copy (a 60 KiB set: 171 us, pinned 180)
    constexpr size_t UP_PIN = 32 << 10;
    if (4 * words <= UP_PIN && !ctx->up_pin &&
        hipHostMalloc((void **)&ctx->up_pin, UP_PIN, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        ctx->up_pin = nullptr;
    }
    const bool pinned = 4 * words <= UP_PIN && ctx->up_pin;
    std::vector<int32_t> pageable;
    int32_t *stage = ctx->up_pin;
    if (pinned) {
        if (ctx->busy && (rc = ctx_hip(ctx, hipStreamSynchronize(ctx->stream), "upload"))) {
            bcx_dgraph_free(ctx, g);
            return rc;
        }
    } else {
        pageable.resize(words);
        stage = pageable.data();
    }
    int32_t *base = (int32_t *)g->pool.p;
    size_t at = 0;
    auto place = [&](const std::vector<int32_t> &v) -> const int32_t * {
        std::copy(v.begin(), v.end(), stage + at);
        const int32_t *p = base + at;
        std::fill(stage + at + v.size(), stage + at + padded(v.size()), 0);
        at += padded(v.size());
        return p;
    };
    for (DComp &dc : g->comps) {
        const HostComp &hc = dc.host;
        dc.dev.n = dc.n;
        dc.dev.arcs = dc.arcs;
        dc.dev.rp = place(hc.rp);
        dc.dev.col = place(hc.col);
        dc.dev.reach = place(hc.reach);
        dc.chains.ptr = place(hc.ch_ptr);
        dc.chains.nodes = place(hc.ch_nodes);
        dc.chains.ends = place(hc.ch_ends);
    }
    if (words && (rc = ctx_hip(ctx, hipMemcpyAsync(g->pool.p, stage, 4 * words, hipMemcpyHostToDevice,
                                                   ctx->stream), "components"))) {
        bcx_dgraph_free(ctx, g);
        return rc;
    }
    ctx->busy = true;
    if (!pinned && (rc = ctx_hip(ctx, hipStreamSynchronize(ctx->stream), "upload"))) {
        bcx_dgraph_free(ctx, g);
        return rc;
    }
    *out = g;
    return BCX_OK;
}

int bcx_batched_order(bcx_ctx *ctx, bcx_dgraph *g, int32_t c, int32_t *order) {
    if (!ctx || !g || !order || c < 0 || c >= (int32_t)g->comps.size()) return BCX_E_ARG;
    const std::vector<int32_t> o = batched_order(g->comps[c]);
    std::memcpy(order, o.data(), sizeof(int32_t) * o.size());
    return BCX_OK;
}

void bcx_dgraph_free(bcx_ctx *ctx, bcx_dgraph *g) {
    if (!g) return;
    if (ctx) {
        if (ctx->busy) (void)hipStreamSynchronize(ctx->stream);
        for (auto &dc : g->comps)
            for (DBuf *b : {&dc.b_rp, &dc.b_col, &dc.b_reach, &dc.b_chp, &dc.b_chn, &dc.b_che, &dc.b_ord}) b->release(ctx);
        batched_graph_release(ctx, g);
        g->pool.release(ctx);
    }
    delete g;
}

// A slice of the BC accumulator that comes back to the host: bc[src, src +
// len) lands at packed[dst, dst + len).
struct BcChunk {
    int64_t src, dst;
    int32_t len, pad;
};
constexpr int32_t BC_CHUNK = 8192;

__global__ void k_bc_gather(const double *bc, double *packed, const BcChunk *ch) {
    const BcChunk c = ch[blockIdx.x];
    for (int i = threadIdx.x; i < c.len; i += blockDim.x) packed[c.dst + i] = bc[c.src + i];
}

constexpr size_t OUT_BYTES = 1 << 20;  // results up to this size may be stored by a kernel

// A result download in flight: the slices that come back and their staging.
struct Download {
    std::vector<BcChunk> chunks;
    std::vector<double> pageable;
    double *stage = nullptr;
};

// Waits for what a failing run has queued, before its host buffers go.
struct Drain {
    bcx_ctx *ctx;
    bool done = false;
    explicit Drain(bcx_ctx *c) : ctx(c) {}
    ~Drain() {
        if (done) return;
        if (ctx->side) (void)hipStreamSynchronize(ctx->side);
        (void)hipStreamSynchronize(ctx->stream);
    }
};

// The slices of a run's BC that come back, and their staging (packed, or as in
// the accumulator); returns their words.  A run over a source subset leaves the
// slices of components without sources at the zeros they were set to, so those
// stay.
static int64_t download_plan(bcx_ctx *ctx, bcx_dgraph *g, const std::vector<char> *touched, Download &d, bool pack) {
    std::vector<BcChunk> &chunks = d.chunks;
    chunks.clear();
    int64_t packed = 0;
    for (size_t ci = 0; ci < g->comps.size(); ++ci) {
        if (touched && !(*touched)[ci]) continue;
        const DComp &dc = g->comps[ci];
        for (int64_t i = 0; i < dc.n; i += BC_CHUNK) {
            BcChunk c{};
            c.src = dc.offset + i;
            c.dst = pack ? packed : c.src;
            c.len = (int32_t)std::min<int64_t>(BC_CHUNK, dc.n - i);
            chunks.push_back(c);
            packed += c.len;
        }
    }
    if (!pack) packed = g->total_n;
    const size_t bytes = sizeof(double) * (size_t)packed;
    if (packed && ctx->bc_pin_bytes < bytes) {
        if (ctx->bc_pin) (void)hipHostFree(ctx->bc_pin);
        ctx->bc_pin = nullptr;
        ctx->bc_pin_bytes = 0;
        if (hipHostMalloc((void **)&ctx->bc_pin, bytes, hipHostMallocDefault) == hipSuccess) {
            ctx->bc_pin_bytes = bytes;
        } else {
            // no pinned memory (a low locked-memory limit): pageable staging
            (void)hipGetLastError();
            ctx->bc_pin = nullptr;
        }
    }
    d.stage = ctx->bc_pin;
    if (!d.stage) {
        d.pageable.resize((size_t)packed);
        d.stage = d.pageable.data();
    }
    return packed;
}

// Starts the copy of the run's BC: gathered into one packed buffer on the device
// and copied to the staging; download_add adds it slice by slice once the stream
// has been waited for.
static int download_start(bcx_ctx *ctx, bcx_dgraph *g, const double *bc, const std::vector<char> *touched, Download &d) {
    const int64_t packed = download_plan(ctx, g, touched, d, true);
    if (packed == 0) return BCX_OK;
    const std::vector<BcChunk> &chunks = d.chunks;
    const size_t bytes = sizeof(double) * (size_t)packed;
    const double *from = bc;
    int rc;
    if (packed < g->total_n) {
        if ((rc = upload(ctx, chunks.data(), sizeof(BcChunk) * chunks.size(), ctx->bc_chunks, "result chunks")) ||
            (rc = ctx->bc_pack.ensure(ctx, bytes, "packed result")))
            return rc;
        hipLaunchKernelGGL(k_bc_gather, dim3((unsigned)chunks.size()), dim3(256), 0, ctx->stream, bc,
                           (double *)ctx->bc_pack.p, (const BcChunk *)ctx->bc_chunks.p);
        if ((rc = ctx_hip(ctx, hipGetLastError(), "result gather"))) return rc;
        from = (const double *)ctx->bc_pack.p;
    }
    return ctx_hip(ctx, hipMemcpyAsync(d.stage, from, bytes, hipMemcpyDeviceToHost, ctx->stream), "bc copy");
}

static void download_add(const Download &d, double *bc_out) {
    for (const BcChunk &c : d.chunks) {
        double *o = bc_out + c.src;
        const double *h = d.stage + c.dst;
        for (int32_t i = 0; i < c.len; ++i) o[i] += h[i];
    }
}

static int run_graph(bcx_ctx *ctx, bcx_dgraph *g, const bcx_opts *opts, double *bc_out, bcx_stats *st, bool copies) {
    if (!ctx || !g) return ctx_fail(ctx, BCX_E_ARG, "null context or graph");
    (void)hipSetDevice(ctx->device);
    bcx_opts o{};
    if (opts) o = *opts;
    if (o.path != BCX_PATH_PLAIN && o.path != BCX_PATH_BATCHED)
        return ctx_fail(ctx, BCX_E_ARG, "unknown path");
    bcx_stats local{};
    bcx_stats *s = st ? st : &local;
    std::memset(s, 0, sizeof(*s));
    auto t0 = std::chrono::steady_clock::now();
    ctx->busy = true;
    ctx->by_source = 0;
    // a run that failed part-way may have left work on the side stream and
    // timer intervals open or uncollected
    batched_persistent_reset(ctx);
    ctx->timer.depth = 0;
    ctx->timer.used = 0;
    ctx->timer_chain.depth = 0;
    ctx->timer_chain.used = 0;
    // subset slots -> per-component local lists
    std::vector<std::vector<int32_t>> sub;
    if (o.src_subset) {
        sub.assign(g->comps.size(), {});
        for (int64_t i = 0; i < o.n_src; ++i) {
            const int64_t slot = o.src_subset[i];
            const size_t ci = (size_t)(std::upper_bound(g->offs.begin(), g->offs.end(), slot) - g->offs.begin());
            if (ci == 0) return ctx_fail(ctx, BCX_E_ARG, "source slot out of range");
            const DComp &dc = g->comps[ci - 1];
            if (slot - dc.offset >= dc.n) return ctx_fail(ctx, BCX_E_ARG, "source slot out of range");
            sub[ci - 1].push_back((int32_t)(slot - dc.offset));
        }
    }
    // the accumulator; for small components with FP64 terms several, where the cap
    // leaves plenty beside them
    const size_t bc_bytes = sizeof(double) * (size_t)std::max<int64_t>(g->total_n, 1);
    int64_t copy = 0;
    if (o.path == BCX_PATH_PLAIN || o.precision != BCX_PREC_FP32C)
        for (size_t ci = 0; ci < g->comps.size() && !copy; ++ci)
            if ((!o.src_subset || !sub[ci].empty()) && src_takes(g->comps[ci], false)) copy = g->total_n;
    if (copy && (!copies || ctx_room(ctx) / 16 < SRC_COPIES * bc_bytes ||
                 ctx->bc_copies.ensure(ctx, SRC_COPIES * bc_bytes, "accumulators") != BCX_OK))
        copy = 0;
    ctx->copies_held = copy != 0;
    struct Held {
        bcx_ctx *ctx;
        ~Held() { ctx->copies_held = false; }
    } held{ctx};
    int rc = copy ? BCX_OK : ctx->bc_acc.ensure(ctx, bc_bytes, "bc accumulator");
    if (rc) return rc;
    double *bc = (double *)(copy ? ctx->bc_copies.p : ctx->bc_acc.p);
    rc = ctx_hip(ctx, hipMemsetAsync(bc, 0, copy ? SRC_COPIES * bc_bytes : bc_bytes, ctx->stream), "memset");
    if (rc) return rc;
    std::vector<SmallJob> srck;   // small components for the wave-per-source kernel (both paths)
    std::vector<SmallJob> small;  // batched path: components for the one-launch small kernel
    std::vector<SmallJob> wg;     // batched path: deep components for the workgroup-per-tile kernel
    std::vector<SmallJob> single;  // batched path: components whose sources run one by one
    std::vector<SmallJob> multi;  // batched path: components for the multi-launch tiles
    int32_t largest_multi = -1;
    for (size_t ci = 0; ci < g->comps.size(); ++ci) {
        DComp &dc = g->comps[ci];
        const int32_t *sp = o.src_subset ? sub[ci].data() : nullptr;
        int64_t sn = o.src_subset ? (int64_t)sub[ci].size() : 0;
        if (o.src_subset && sn == 0) continue;
        // algorithmic work of the reference's method: BFS sources (free and
        // chain endpoints) and chain sources
        auto account = [&](int64_t n_bfs, int64_t n_chain) {
            s->n_bfs_sources += n_bfs;
            s->n_chain_sources += n_chain;
            s->bytes_alg += (double)n_bfs * (16.0 * dc.arcs + 80.0 * dc.n) +
                            (double)n_chain * (8.0 * dc.arcs + 100.0 * dc.n);
            s->teps_work += (double)(n_bfs + n_chain) * (double)dc.arcs * 0.5;
        };
        if (o.path == BCX_PATH_PLAIN && o.row_cap_bytes <= 0 && src_takes(dc, false) &&
            plain_scratch_fits(ctx, dc.n, sp ? sn : dc.n)) {
            // every source runs on its own, chain vertices included: with the
            // state in LDS a traversal costs less than the combine of two
            // endpoint rows (a caller who sizes the row slab gets the rows,
            // and a cap below the per-source rows is refused as before)
            std::vector<uint8_t> want((size_t)dc.n, sp ? 0 : 1);
            for (int64_t i = 0; i < sn; ++i) want[(size_t)sp[i]] = 1;
            std::vector<int32_t> srcs;
            for (int32_t v = 0; v < dc.n; ++v)
                if (want[(size_t)v]) srcs.push_back(v);
            int64_t n_chain = 0;
            if (o.use_chains)
                for (int32_t v : dc.host.ch_nodes) n_chain += want[(size_t)v];
            account((int64_t)srcs.size() - n_chain, n_chain);
            srck.push_back({&dc, std::move(srcs)});
            continue;
        }
        if (o.path == BCX_PATH_PLAIN) {
            Plan plan;
            // (a caller who sizes the row slab gets the rows)
            rc = make_plan(dc.host, sp, sn, o.use_chains != 0, row_capacity(ctx, dc.n, &o), o.row_cap_bytes <= 0, plan);
            if (rc) return rc;
            account(plan.n_bfs, plan.n_chain);
            s->n_row_only += plan.n_row_only;
            rc = plain_component(ctx, dc, plan, &o, bc + dc.offset, s);
            if (rc) return rc;
            continue;
        }
        int64_t n_chain = 0;
        std::vector<int32_t> srcs = batched_sources(dc, sp, sn, o.use_chains ? &n_chain : nullptr);
        account((int64_t)srcs.size() - n_chain, n_chain);
        const int kind = batched_schedule(ctx, dc, &o, (int64_t)srcs.size(), s);  // (one-time sample runs stay outside the timing)
        if (kind < 0) return kind;
        if (kind == BCX_KERNEL_SMALL) {
            s->n_comp_small++;
            (src_takes(dc, o.precision == BCX_PREC_FP32C) ? srck : small).push_back({&dc, std::move(srcs)});
            continue;
        }
        // larger components: tile order from the tuner (BFS ranks or balls); run
        // source by source, the sources keep theirs (ordering 16384 sources of a
        // 26k grid in balls took 1.7 ms of the run's 25.9)
        tune_order(dc);
        std::vector<int32_t> tiles = kind == KIND_SOURCE ? std::move(srcs) : tuned_sources(dc, srcs);
        if (dc.tile_order == 1) s->n_ball_tiles++;
        if (kind == BCX_KERNEL_WG || kind == KIND_SOURCE) {
            s->n_comp_wg++;
            (kind == KIND_SOURCE ? single : wg).push_back({&dc, std::move(tiles)});
        } else {
            const bcx_opts own = batched_opts(dc, o);
            if ((rc = batched_prepare(ctx, dc, &own))) return rc;  // one-time work stays outside the timing
            s->n_comp_multi++;
            if (dc.n > largest_multi) {
                largest_multi = dc.n;
                batched_sched_report(dc, &o, &s->sched_blocks_per_cu, &s->sched_slots, &s->sched_sources_per_lane);
            }
            multi.push_back({&dc, std::move(tiles)});
        }
    }
    std::vector<char> touched;
    if (o.src_subset) {
        touched.assign(g->comps.size(), 0);
        for (size_t ci = 0; ci < g->comps.size(); ++ci) touched[ci] = !sub[ci].empty();
    }
    const bool want = bc_out && g->total_n > 0;
    Download down;
    Drain drain(ctx);
    bool downloaded = false;
    if (!srck.empty() && small.empty() && wg.empty() && single.empty() && multi.empty()) {
        // the one-launch pass alone: its counters and the result come back
        // behind it and the host waits once (with two more waits and a pageable
        // upload a 24-vertex call takes 88 us, so 75)
        // With several accumulators, the kernel that adds them up stores a small
        // result in the pinned buffer itself, in place of the two copies (host call
        // of four blocks of 600 vertices: 152 us with one accumulator, 187 with
        // that launch before the copies, 146 so; of 24 vertices 75 and 48).
        double *out = nullptr;
        const std::vector<char> *some = o.src_subset ? &touched : nullptr;
        if (want && copy && bc_bytes <= OUT_BYTES) {
            (void)download_plan(ctx, g, some, down, false);
            if (down.pageable.empty()) out = down.stage;
        }
        ctx->timer.begin(ctx);
        rc = batched_persistent_start(ctx, srck, &o, bc, s, PASS_SRC, ctx->stream, copy, out);
        ctx->timer.end(ctx);
        if (rc || (want && !out && (rc = download_start(ctx, g, bc, some, down)))) return rc;
        bool again = false;
        if ((rc = batched_persistent_finish(ctx, s, PASS_SRC, &again))) return rc;
        downloaded = want && !again;
    } else if (!srck.empty() || !small.empty() || !wg.empty() || !single.empty() || !multi.empty()) {
        // the persistent passes (small components, deep components) run on a
        // side stream while the multi-launch tiles run on theirs; the run is
        // timed as one interval on the context stream around both
        const bool overlap = (!multi.empty() || !single.empty()) && (!srck.empty() || !small.empty() || !wg.empty());
        if (overlap && !ctx->side &&
            (rc = ctx_hip(ctx, hipStreamCreateWithFlags(&ctx->side, hipStreamNonBlocking), "side stream")))
            return rc;
        const hipStream_t sp = overlap ? ctx->side : ctx->stream;
        ctx->timer.begin(ctx);
        if ((rc = batched_persistent_start(ctx, srck, &o, bc, s, PASS_SRC, sp, copy)) ||
            (rc = batched_persistent_start(ctx, small, &o, bc, s, PASS_SMALL, sp)) ||
            (rc = batched_persistent_start(ctx, wg, &o, bc, s, PASS_WG, sp)))
            return rc;
        for (SmallJob &jb : multi) {
            DComp &dc = *const_cast<DComp *>(jb.dc);
            const bcx_opts own = batched_opts(dc, o);
            if ((rc = batched_component(ctx, dc, jb.srcs, &own, bc + dc.offset, s))) return rc;
        }
        std::vector<SmallJob> again;  // FP32 terms with overflowed counts, or no room for rows beside the tiles
        for (SmallJob &jb : single) {
            bool overflow = false;
            rc = source_component(ctx, *const_cast<DComp *>(jb.dc), jb.srcs, &o, bc + jb.dc->offset, s, &overflow);
            if (rc && rc != BCX_E_NOMEM) return rc;
            if (rc || overflow) again.push_back(std::move(jb));  // (nothing was added)
            else ctx->by_source++;
        }
        if ((rc = batched_persistent_finish(ctx, s, PASS_SRC)) || (rc = batched_persistent_finish(ctx, s, PASS_SMALL)) ||
            (rc = batched_persistent_finish(ctx, s, PASS_WG)))
            return rc;
        for (SmallJob &jb : again) {
            // (in the order of the tiles: those around an overflow turn to FP64)
            DComp &dc = *const_cast<DComp *>(jb.dc);
            const std::vector<SmallJob> tiles{{&dc, tuned_sources(dc, jb.srcs)}};
            if (dc.n > WG_N) {
                const bcx_opts own = batched_opts(dc, o);
                if ((rc = batched_prepare(ctx, dc, &own)) ||
                    (rc = batched_component(ctx, dc, tiles[0].srcs, &own, bc + dc.offset, s)))
                    return rc;
                continue;
            }
            if ((rc = batched_persistent_start(ctx, tiles, &o, bc, s, PASS_WG, ctx->stream)) ||
                (rc = batched_persistent_finish(ctx, s, PASS_WG)))
                return rc;
        }
        if (overlap) {
            hipEvent_t ev;
            if ((rc = ctx_hip(ctx, hipEventCreateWithFlags(&ev, hipEventDisableTiming), "event"))) return rc;
            rc = ctx_hip(ctx, hipEventRecord(ev, sp), "event");
            if (!rc) rc = ctx_hip(ctx, hipStreamWaitEvent(ctx->stream, ev, 0), "event");
            (void)hipEventDestroy(ev);
            if (rc) return rc;
        }
        ctx->timer.end(ctx);
    }
    if (!downloaded) {
        if (want && (rc = download_start(ctx, g, bc, o.src_subset ? &touched : nullptr, down))) return rc;
        if ((rc = ctx_hip(ctx, hipStreamSynchronize(ctx->stream), "run"))) return rc;
    }
    drain.done = true;
    if (want) download_add(down, bc_out);
    ctx->busy = false;
    s->t_chain_s = ctx->timer_chain.collect();
    s->t_kernel_s = ctx->timer.collect() + s->t_chain_s;
    s->t_total_s = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    return BCX_OK;
}

int bcx_run(bcx_ctx *ctx, bcx_dgraph *g, const bcx_opts *opts, double *bc_out, bcx_stats *st) {
    int rc = run_graph(ctx, g, opts, bc_out, st, true);
    if (rc == BCX_E_NOMEM && ctx->bc_copies.p) {  // (nothing was added to bc_out)
        ctx->bc_copies.release(ctx);
        rc = run_graph(ctx, g, opts, bc_out, st, false);
    }
    return rc;
}

int32_t bcx_run_by_source(const bcx_ctx *ctx) { return ctx ? ctx->by_source : 0; }

int bcx_bc(bcx_ctx *ctx, const bcx_component *comps, int32_t n_comps, const bcx_opts *opts,
           double *bc_out, bcx_stats *st) {
    bcx_dgraph *g = nullptr;
    int rc = bcx_upload(ctx, comps, n_comps, &g);
    if (rc) return rc;
    rc = bcx_run(ctx, g, opts, bc_out, st);
    bcx_dgraph_free(ctx, g);
    return rc;
}

int bcx_host_bc(bcx_ctx *ctx, const bcx_host *h, const bcx_opts *opts, double *bc_out, bcx_stats *st) {
    if (!ctx || !h || !bc_out || !h->decomposed) return ctx_fail(ctx, BCX_E_ARG, "host graph not decomposed");
    std::vector<bcx_component> comps;
    int64_t total = 0;
    for (auto &c : h->comps) { comps.push_back(c.view()); total += c.n; }
    std::vector<double> local((size_t)std::max<int64_t>(total, 1), 0.0);
    int rc = BCX_OK;
    if (!comps.empty()) rc = bcx_bc(ctx, comps.data(), (int32_t)comps.size(), opts, local.data(), st);
    if (rc) return rc;
    for (int32_t v = 0; v < h->n; ++v) bc_out[v] = (double)h->cut[v];
    int64_t off = 0;
    for (auto &c : h->comps) {
        for (int32_t i = 0; i < c.n; ++i) bc_out[c.gid[i]] += local[off + i];
        off += c.n;
    }
    return BCX_OK;
}

int bcx_debug_source(bcx_ctx *ctx, const bcx_component *comp, int32_t src, const bcx_opts *opts,
                     int32_t *level, uint64_t *sigma_u64, double *sigma_f64, double *delta,
                     int32_t *sigma_is_f64) {
    if (!ctx || !comp || src < 0 || src >= comp->n) return ctx_fail(ctx, BCX_E_ARG, "bad debug args");
    bcx_opts o{};
    if (opts) o = *opts;
    if (o.path == BCX_PATH_BATCHED)
        return batched_debug_tile(ctx, comp, &src, 1, &o, level, sigma_u64, sigma_f64, delta, sigma_is_f64, nullptr);
    bcx_dgraph *g = nullptr;
    int rc = bcx_upload(ctx, comp, 1, &g);
    if (rc) return rc;
    DComp &dc = g->comps[0];
    const int32_t n = dc.n;
    std::vector<int32_t> lv(n);
    std::vector<uint64_t> sg(n);
    std::vector<double> dl(n);
    bool f64 = false;
    const uint64_t limit = (o.sigma_f64_threshold_log2 > 0 && o.sigma_f64_threshold_log2 < 64)
                               ? (1ull << o.sigma_f64_threshold_log2) : 0;
    // is src a chain vertex?
    int32_t ci = -1, pos = -1;
    if (o.use_chains)
        for (int32_t c = 0; c < dc.host.n_chains && ci < 0; ++c)
            for (int32_t j = dc.host.ch_ptr[c]; j < dc.host.ch_ptr[c + 1]; ++j)
                if (dc.host.ch_nodes[j] == src) { ci = c; pos = j - dc.host.ch_ptr[c]; break; }
    rc = ctx->bc_acc.ensure(ctx, sizeof(double) * n, "bc accumulator");
    DBuf probe;
    if (!rc) rc = probe.ensure(ctx, 2 * sizeof(double) * (size_t)n, "probe delta");
    for (int attempt = 0; attempt < 2 && !rc; ++attempt) {
        ctx->overflow = false;
        Rows rows{};
        if ((rc = ensure_rows(ctx, n, 2, rows))) break;
        PlainScratch sc;
        double *bc = (double *)ctx->bc_acc.p, *pd = (double *)probe.p;
        if ((rc = ctx_hip(ctx, hipMemsetAsync(pd, 0, sizeof(double) * (size_t)n, ctx->stream), "memset"))) break;
        if (ci < 0) {
            std::vector<int32_t> s{src}, sl{0};
            std::vector<int8_t> m{(int8_t)(MODE_BC | MODE_ROW)};
            rc = run_bfs_list(ctx, dc, s, sl, m, f64, limit, bc, rows, nullptr, pd);
            if (rc) break;
            if (ctx->overflow && !f64) { f64 = true; continue; }
            rc = ctx_hip(ctx, hipMemcpyAsync(lv.data(), rows.d, 4 * n, hipMemcpyDeviceToHost, ctx->stream), "copy");
            if (!rc) rc = ctx_hip(ctx, hipMemcpyAsync(sg.data(), rows.sig, 8 * n, hipMemcpyDeviceToHost, ctx->stream), "copy");
        } else {
            std::vector<int32_t> s{dc.host.ch_ends[2 * ci], dc.host.ch_ends[2 * ci + 1]}, sl{0, 1};
            std::vector<int8_t> m{MODE_ROW, MODE_ROW};
            rc = run_bfs_list(ctx, dc, s, sl, m, f64, limit, bc, rows, nullptr);
            if (rc) break;
            if (ctx->overflow && !f64) { f64 = true; continue; }
            PlanBatch b;
            b.cci = {ci};
            b.cpos = {pos};
            b.cslots = {0, 1};
            rc = run_chain_list(ctx, dc, b, f64, bc, rows, nullptr, pd);
            if (rc) break;
            // the chain launch ran one workgroup: its rows start at offset 0
            if ((rc = ensure_plain_scratch(ctx, n, 1, sc))) break;
            rc = ctx_hip(ctx, hipMemcpyAsync(lv.data(), sc.d, 4 * n, hipMemcpyDeviceToHost, ctx->stream), "copy");
            if (!rc) rc = ctx_hip(ctx, hipMemcpyAsync(sg.data(), sc.sig, 8 * n, hipMemcpyDeviceToHost, ctx->stream), "copy");
        }
        if (!rc) rc = ctx_hip(ctx, hipMemcpyAsync(dl.data(), pd, 8 * n, hipMemcpyDeviceToHost, ctx->stream), "copy");
        if (!rc) rc = ctx_hip(ctx, hipStreamSynchronize(ctx->stream), "copy");
        break;
    }
    (void)ctx->timer.collect();
    (void)ctx->timer_chain.collect();
    probe.release(ctx);
    bcx_dgraph_free(ctx, g);
    if (rc) return rc;
    dl[src] = 0.0;
    if (level) std::memcpy(level, lv.data(), 4 * n);
    for (int32_t i = 0; i < n; ++i) {
        if (sigma_u64) sigma_u64[i] = f64 ? 0 : sg[i];
        double f;
        std::memcpy(&f, &sg[i], 8);
        if (sigma_f64) sigma_f64[i] = f64 ? f : (double)sg[i];
    }
    if (delta) std::memcpy(delta, dl.data(), 8 * n);
    if (sigma_is_f64) *sigma_is_f64 = f64 ? 1 : 0;
    return BCX_OK;
}

int bcx_debug_tile(bcx_ctx *ctx, const bcx_component *comp, const int32_t *srcs, int32_t ns, const bcx_opts *opts,
                   int32_t *level, uint64_t *sigma_u64, double *sigma_f64, double *delta, int32_t *sigma_is_f64,
                   int32_t *kernel_used) {
    if (!ctx || !comp || !srcs || ns < 1 || ns > BATCH_W * MAX_SPL || comp->n <= 0)
        return ctx_fail(ctx, BCX_E_ARG, "bad debug tile args");
    std::vector<uint8_t> seen((size_t)comp->n, 0);
    for (int32_t i = 0; i < ns; ++i) {
        if (srcs[i] < 0 || srcs[i] >= comp->n || seen[(size_t)srcs[i]])
            return ctx_fail(ctx, BCX_E_ARG, "tile sources must be distinct vertices of the component");
        seen[(size_t)srcs[i]] = 1;
    }
    (void)hipSetDevice(ctx->device);
    ctx->busy = true;
    bcx_opts o{};
    if (opts) o = *opts;
    return batched_debug_tile(ctx, comp, srcs, ns, &o, level, sigma_u64, sigma_f64, delta, sigma_is_f64,
                              kernel_used);
}

}  // extern "C"
