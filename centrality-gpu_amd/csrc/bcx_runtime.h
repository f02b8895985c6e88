// Runtime types shared by the plain and batched host drivers.
#pragma once
#include <hip/hip_runtime.h>

#include <array>
#include <map>
#include <string>
#include <utility>
#include <vector>

#include "bcx.h"
#include "bcx_device.h"
#include "bcx_kernels.h"

struct bcx_ctx;

namespace bcx {

// Grow-only device buffer accounted against the context's memory cap.
struct DBuf {
    void *p = nullptr;
    size_t bytes = 0;
    int ensure(bcx_ctx *ctx, size_t need, const char *what);
    void release(bcx_ctx *ctx);
};

// HIP-event intervals on the context stream, summed by collect().  Nested
// begin/end pairs record only at the outermost level, so a run whose
// streams overlap is timed as one interval.
struct Timer {
    std::vector<std::pair<hipEvent_t, hipEvent_t>> evs;
    size_t used = 0;
    int depth = 0;
    void begin(bcx_ctx *ctx);
    void end(bcx_ctx *ctx);
    double collect();
    void destroy();
};

// Host copy of a component (planning needs the chains and the degrees).
struct ChainCut;  // multi-launch copy with contracted chains (bcx_batched_host.hip)

struct HostComp {
    int32_t n = 0;
    int64_t arcs = 0;
    std::vector<int32_t> rp, col, reach;
    int32_t n_chains = 0;
    std::vector<int32_t> ch_ptr, ch_nodes, ch_ends;
};

// Seconds measured on a component (negative: not yet), under the options of
// `key` (FP32C, chains contracted, sources per lane, tiles in flight, blocks
// per CU).
struct KindTimes {
    std::array<int32_t, 5> key{};
    double src = -1.0;   // a source on the per-source kernel, of a full launch
    double tile = -1.0;  // a multi-launch tile alone
    double more = -1.0;  // each source past its own
    double wg = -1.0;    // a round of the workgroup kernel's tiles
};

struct DComp {
    int32_t n = 0;
    int64_t arcs = 0;
    int64_t offset = 0;  // into the concatenated BC vector
    int32_t depth = -1;  // BFS depth from the highest-degree vertex (-1: not measured)
    int32_t core_depth = 0;  // deepest of its levels off the chains (measured with depth)
    double round_ms = -1.0;  // batched path: a round of workgroup tiles, estimated (-1: not yet)
    double sigma_est = 0.0;  // largest path count of that BFS (measured with depth)
    bool src_wrapped = false;  // a per-source FP32C run met counts past 64 bits
    std::vector<int32_t> rank;      // batched path: BFS rank of each vertex (built on first use)
    std::vector<uint8_t> on_chain;  // batched path: 1 for chain vertices (built on first use)
    std::vector<int32_t> ball;      // batched path: every vertex in ball-tile order (built on first use)
    int8_t tile_order = -1;         // batched path: 0 BFS-rank, 1 ball, 2 landmark tiles (tuned on first use)
    std::vector<int32_t> lm_pos;    // batched path: position of each vertex in the landmark order
    int64_t groups = 0;             // sum over the rows of ceil(arcs / 4) (wave-per-source kernel)
    HostComp host;
    DBuf b_rp, b_col, b_reach, b_chp, b_chn, b_che;
    CompDev dev{};
    ChainDev chains{};
    // multi-launch batched path: the component relabelled in BFS order from
    // its highest-degree vertex (built on first use), perm[new] = old on the
    // device, inv[old] = new
    DComp *relabel = nullptr;
    DBuf b_perm;
    std::vector<int32_t> relabel_inv;
    // per-source kernel: the component in BFS order from its highest-degree
    // vertex (built on first use; ord_state -1 not yet looked at, 0 degrees too
    // even, 1 built), ord_inv[old] = new, ord_perm[new] = old
    int8_t ord_state = -1;
    CompDev ord{};
    DBuf b_ord;
    const int32_t *ord_perm = nullptr;
    std::vector<int32_t> ord_inv;
    // multi-launch batched path with contracted chains (built on first use;
    // cut_state -1 not yet tried, 0 the component has too few such chains)
    ChainCut *cut = nullptr;
    int8_t cut_state = -1;
    // FP32C: rounding of the component's terms without and with chains to
    // contract (FP32_ROWS or FP32_TILES; -1 not yet looked at)
    int8_t fp32_route[2] = {-1, -1};
    // batched path: what was measured on sample sources, cached for every later
    // run under the same options (sched_multi: the multi-launch fields below were)
    std::vector<KindTimes> times;
    bool sched_multi = false;
    int8_t sched_cut = 1;     // multi-launch: 1 contracted chains, 0 the relabelled copy
    int16_t sched_bpc = 0;    // multi-launch: level-kernel blocks per CU (0: default)
    int16_t sched_slots = 0;  // multi-launch: tiles in flight (0: default)
    int8_t sched_spl = 0;     // multi-launch: sources per lane, 1, 2 or 4 (0: default)
};

// One endpoint-row batch: BFS work (endpoints, with slot and mode) then the
// chain sources that combine those rows.
struct PlanBatch {
    std::vector<int32_t> bsrc, bslot;
    std::vector<int8_t> bmode;
    std::vector<int32_t> cci, cpos, cslots;
    int32_t n_rows = 0;
};

struct Plan {
    std::vector<int32_t> free_src;     // BFS sources that need no row
    std::vector<PlanBatch> batches;
    // sources by their role in the method: n_chain counts the chain vertices,
    // those among free_src too
    int64_t n_bfs = 0, n_chain = 0, n_row_only = 0;
};

int make_plan(const HostComp &hc, const int32_t *subset, int64_t n_sub, bool use_chains,
              int64_t row_cap, bool direct, Plan &plan);

}  // namespace bcx

struct BatchedState;  // batched path buffers (bcx_batched_host.hip)
struct SmallState;    // small-component kernel buffers (bcx_batched_host.hip)

struct bcx_ctx {
    int device = 0;
    int n_cu = 0;
    std::string name;
    size_t mem_cap = 0, mem_used = 0;
    std::map<void *, size_t> sizes;
    hipStream_t stream = nullptr;
    hipStream_t side = nullptr;  // batched: persistent passes beside the multi-launch tiles
    std::string err;
    bool overflow = false;
    bcx::Timer timer, timer_chain;
    bcx::DBuf counters, bc_acc, plain_scratch, rows_buf;
    bcx::DBuf w_src, w_aux, w_mode, w_slots, bc_split;
    bcx::DBuf bc_pack, bc_chunks;  // result download: packed slices and their chunk list
    double *bc_pin = nullptr;      // pinned host staging of the result download
    size_t bc_pin_bytes = 0;
    int32_t *up_pin = nullptr;     // pinned host staging of small uploads
    bcx::DBuf bc_copies;           // accumulators of a run with several (see SrcArgs::copy)
    bool copies_held = false;      // a run is using them
    int rows_held = 0;             // plain_scratch and bc_split belong to a launch being put together
    int32_t by_source = 0;         // batched: components the last run took source by source
    bool busy = true;              // work may be in flight on the context stream
    BatchedState *batched = nullptr;
    SmallState *small = nullptr;
    SmallState *wgk = nullptr;  // workgroup-per-tile kernel buffers
    SmallState *srck = nullptr;  // wave-per-source kernel buffers
    std::vector<bcx::DBuf *> all_bufs() {
        return {&counters, &bc_acc, &plain_scratch, &rows_buf, &w_src, &w_aux, &w_mode, &w_slots, &bc_split, &bc_copies, &bc_pack, &bc_chunks};
    }
};

struct bcx_dgraph {
    std::vector<bcx::DComp> comps;
    std::vector<int64_t> offs;  // comps[i].offset, packed for the source-slot search
    int64_t total_n = 0;
    bcx::DBuf pool;  // every component's CSR, reach and chain arrays, one allocation
};

// shared helpers (bcx_runtime.hip)
int ctx_fail(bcx_ctx *ctx, int code, const std::string &msg);
int ctx_hip(bcx_ctx *ctx, hipError_t e, const char *what);
int dev_alloc(bcx_ctx *ctx, void **p, size_t bytes, const char *what);
void dev_free(bcx_ctx *ctx, void *p);
// Device memory that allocations can still get under the cap (what the idle
// rows of the per-source kernel hold is given back for them).
size_t ctx_room(const bcx_ctx *ctx);
int upload(bcx_ctx *ctx, const void *host, size_t bytes, bcx::DBuf &buf, const char *what);
int read_counters(bcx_ctx *ctx, bcx_stats *st);
int64_t row_capacity(bcx_ctx *ctx, int32_t n, const bcx_opts *o);
int plain_component(bcx_ctx *ctx, bcx::DComp &dc, const bcx::Plan &plan, const bcx_opts *o,
                    double *bc, bcx_stats *st);

// Device address of the no-allocation entry point's static scratch array on
// `device` (current), looked up once per device (bcx_noalloc.hip).
int noalloc_init(int device);

// batched path (bcx_batched_host.hip)
struct SmallJob {
    const bcx::DComp *dc;
    std::vector<int32_t> srcs;
};
std::vector<int32_t> batched_sources(bcx::DComp &dc, const int32_t *subset, int64_t n_sub, int64_t *n_chain);
std::vector<int32_t> ball_sources(bcx::DComp &dc, const std::vector<int32_t> &srcs);
void tune_order(bcx::DComp &dc);
std::vector<int32_t> tuned_sources(bcx::DComp &dc, const std::vector<int32_t> &srcs);
// Every vertex of the component in the order a full batched run tiles its
// sources (64 consecutive entries per tile).
std::vector<int32_t> batched_order(bcx::DComp &dc);
// One persistent launch over the tiles of `jobs`, started on stream sp
// without waiting; _finish waits for it and reruns overflowed tiles in FP64.
// The passes: 64-source tiles of small components, the workgroup-per-tile
// kernel, and the wave-per-source kernel (components that src_takes accepts;
// copy: words from one of its zeroed accumulators to the next, 0: there is one;
// out: pinned buffer for the sums of every component, with copy only).
enum { PASS_SMALL = 0, PASS_WG = 1, PASS_SRC = 2 };
int batched_persistent_start(bcx_ctx *ctx, const std::vector<SmallJob> &jobs, const bcx_opts *o, double *bc_base,
                             bcx_stats *st, int pass, hipStream_t sp, int64_t copy = 0,
                             double *out = nullptr);
// (*again, optional: some of it was rerun after the first launch)
int batched_persistent_finish(bcx_ctx *ctx, bcx_stats *st, int pass, bool *again = nullptr);
// Whether the wave-per-source kernel takes a component, with FP32 or FP64 terms.
bool src_takes(const bcx::DComp &dc, bool fp32);
// Drops passes left unfinished by an earlier failed run (after waiting for them).
void batched_persistent_reset(bcx_ctx *ctx);
bool batched_narrow(bcx::DComp &dc);
void small_release(bcx_ctx *ctx);
// One-time preparation of a multi-launch component (its relabelled copy, or
// the copy with contracted chains when the options ask for chains).
int batched_prepare(bcx_ctx *ctx, bcx::DComp &dc, const bcx_opts *o);
int batched_component(bcx_ctx *ctx, bcx::DComp &dc, const std::vector<int32_t> &srcs, const bcx_opts *o,
                      double *bc, bcx_stats *st);
// Kernel (BCX_KERNEL_*) the batched path runs a component on, given the
// bcx_opts flags.
int batched_kind(bcx::DComp &dc, int flags);
// The kernel and, for the multi-launch tiles, the schedule of a component of
// the batched path: measured once on sample tiles for components of at least
// TUNE_N vertices (unless the options fix it), else batched_kind's rule.
// Returns a BCX_KERNEL_*, KIND_SOURCE (the per-source kernel of the plain path,
// sources one by one) or a negative BCX_E_* status.
constexpr int KIND_SOURCE = 4;
int batched_schedule(bcx_ctx *ctx, bcx::DComp &dc, const bcx_opts *o, int64_t n_src, bcx_stats *st);
// The sources srcs of a component on the per-source kernel in the run's
// precision.  *overflow: a uint64 count overflowed with FP32 terms; bc is as
// before and the component is left to the tiled kernels, which turn to FP64
// terms tile by tile.
int source_component(bcx_ctx *ctx, bcx::DComp &dc, const std::vector<int32_t> &srcs, const bcx_opts *o, double *bc,
                     bcx_stats *st, bool *overflow);
// Whether the context's cap leaves room for the per-source kernel's rows.
bool plain_scratch_fits(bcx_ctx *ctx, int32_t n, int64_t count);
// The options that a component's multi-launch tiles run under, once it has its
// schedule: FP32C runs round the terms of a component alike in every call.
bcx_opts batched_opts(const bcx::DComp &dc, const bcx_opts &o);
// Blocks per CU, tiles in flight and sources per lane a multi-launch run of
// dc uses.
void batched_sched_report(const bcx::DComp &dc, const bcx_opts *o, int32_t *bpc, int32_t *slots, int32_t *spl);
int batched_debug_tile(bcx_ctx *ctx, const bcx_component *comp, const int32_t *srcs, int32_t ns, const bcx_opts *o,
                       int32_t *level, uint64_t *sigma_u64, double *sigma_f64, double *delta, int32_t *sigma_is_f64,
                       int32_t *kernel_used);
void batched_release(bcx_ctx *ctx);
void batched_graph_release(bcx_ctx *ctx, bcx_dgraph *g);
