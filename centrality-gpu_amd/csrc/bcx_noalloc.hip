// bcx_bc_small_noalloc: the batched run of one small component (n <=
// BCX_NOALLOC_MAX_N) on the small-component kernels, with every buffer beyond
// the caller's inputs and output in one static device array, so the call
// allocates nothing.  The launch sequence is kernels only:
//   setup   tile tables, sources, weights, zeroed counters and accumulators,
//           validity check, which kernel the component fits
//   k_src   a wave per source, 64-bit path counts, into the array's own BC: 16
//           accumulators, so that the sum over many small tiles is as accurate
//           as over 64-source ones (1000 sources, error against 64 bits: one
//           accumulator 4.4e-16, k_small 1.8e-16)
//   add     their sum, rounded once, into the caller's when no count left 64 bits
// followed by one read-back of the status words and a stream sync.  Components
// with too many arcs for the LDS of k_src, and those with a count past 64 bits
// (whose 64-source tiles turn to FP64 counts and terms as in bcx_run), go on:
//   k_small 64-bit path counts over every tile (tile count read on device)
//   remap   the tiles whose counts left 64 bits become the second table
//   k_small FP64 path counts over those tiles (none: returns at once)
// k_src holds its state in LDS, so its workgroups are not bound by the array's
// slabs: a 1000-vertex component of average degree 8, every source: 2.48 ms on
// 8 workgroups of k_small, 0.13 ms on 250 of k_src (the whole call).
#include <algorithm>
#include <mutex>
#include <string>

#include "bcx.h"
#include "bcx_runtime.h"
#include "bcx_small.h"
#include "bcx_src.h"

using namespace bcx;

namespace {

constexpr int NA_N = BCX_NOALLOC_MAX_N;
constexpr int NA_WG = BCX_NOALLOC_MAX_WORKGROUPS;
constexpr int NA_TILES = (NA_N + 63) / 64;
constexpr int NA_STILES = 256;  // tiles of k_src: few sources each, to use every compute unit
constexpr int NA_COPIES = 16;   // accumulators of k_src
constexpr size_t NA_SLAB = (size_t)NA_N * 64;  // words per workgroup slab
static_assert(NA_N <= SMALL_N, "the small-component kernel's LDS holds SMALL_N vertices");

constexpr size_t up(size_t x) { return (x + 255) & ~(size_t)255; }

// byte offsets of the scratch array's parts
constexpr size_t O_COMP = 0;
constexpr size_t O_TILES1 = up(O_COMP + sizeof(SmallComp));
constexpr size_t O_TILES2 = up(O_TILES1 + sizeof(SmallTile) * NA_TILES);
constexpr size_t O_SRCS = up(O_TILES2 + sizeof(SmallTile) * NA_TILES);
constexpr size_t O_WS = up(O_SRCS + 4 * (size_t)NA_N);
constexpr size_t O_ZERO = up(O_WS + 8 * (size_t)NA_N);
constexpr size_t O_CTR = up(O_ZERO + 4 * (size_t)NA_N);
constexpr size_t O_REDO1 = up(O_CTR + 64);
constexpr size_t O_REDO2 = up(O_REDO1 + 4 * (size_t)NA_TILES);
constexpr size_t O_COMP0 = up(O_REDO2 + 4 * (size_t)NA_TILES);
constexpr size_t O_TILES0 = up(O_COMP0 + sizeof(SmallComp) * NA_COPIES);
constexpr size_t O_REDO0 = up(O_TILES0 + sizeof(SmallTile) * NA_STILES);
constexpr size_t O_SIG = up(O_REDO0 + 4 * (size_t)NA_STILES);
constexpr size_t O_BC = O_SIG;  // (k_src's accumulators, before k_small uses the slabs)
static_assert((size_t)NA_COPIES * NA_N <= NA_SLAB * NA_WG, "the accumulators fit in the slabs");
constexpr size_t O_TT = O_SIG + 8 * NA_SLAB * NA_WG;
constexpr size_t O_Q = O_TT + 8 * NA_SLAB * NA_WG;
constexpr size_t O_QM = O_Q + 4 * NA_SLAB * NA_WG;
constexpr size_t O_END = O_QM + 8 * NA_SLAB * NA_WG;
static_assert(O_END <= BCX_NOALLOC_SCRATCH_BYTES, "scratch layout exceeds the stated size");

// status words at O_CTR: [0..3] first k_small pass counters, [4..7] second pass
// counters, [8] first pass tiles, [9] second pass tiles, [10] invalid input,
// [11] k_src tiles, [12..14] k_src counters
enum { C1 = 0, C2 = 4, N1 = 8, N2 = 9, BAD = 10, N0 = 11, C0 = 12 };

struct NaArgs {
    int32_t n, n_src, n_tiles, n_stiles, stile;  // 64-source tiles; tiles of k_src and their sources
    int32_t lds;                                 // k_src's dynamic LDS (0: not to be used)
    int32_t min_waves;
    const int32_t *rp, *col, *reach, *srcs;
    double *bc;
    unsigned char *base;  // the scratch array's device address
};

}  // namespace

// The scratch array.  Host code must use its device address from
// hipGetSymbolAddress (kept per device below), never this name.
static __device__ __align__(256) unsigned char scratch[BCX_NOALLOC_SCRATCH_BYTES];

static std::mutex g_mu;
static void *g_ptr[64];      // device address of `scratch` per device
static hipError_t g_err[64];  // result of the lookup per device

// Set-up, from bcx_create with `device` current: looks the array's device
// address up once per device.
int noalloc_init(int device) {
    if (device < 0 || device >= 64) return BCX_E_ARG;
    std::lock_guard<std::mutex> lk(g_mu);
    if (g_ptr[device]) return BCX_OK;
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    g_err[device] = e;
    if (e != hipSuccess || !p) return BCX_E_HIP;
    g_ptr[device] = p;
    return BCX_OK;
}

// (launched with 1 + NA_COPIES blocks: the first sets up, the others clear an
// accumulator each)
__global__ __launch_bounds__(256) void k_na_setup(NaArgs x) {
    unsigned char *b = x.base;
    double *bc0 = (double *)(b + O_BC);
    if (blockIdx.x > 0) {
        for (int v = threadIdx.x; v < x.n; v += blockDim.x) bc0[(int)(blockIdx.x - 1) * NA_N + v] = 0.0;
        return;
    }
    int32_t *ctr = (int32_t *)(b + O_CTR);
    int32_t *srcs = (int32_t *)(b + O_SRCS);
    double *ws = (double *)(b + O_WS);
    int32_t *zero = (int32_t *)(b + O_ZERO);
    SmallTile *tiles = (SmallTile *)(b + O_TILES1);
    __shared__ int bad, groups;
    if (threadIdx.x == 0) bad = groups = 0;
    __syncthreads();
    int g = 0;
    for (int v = threadIdx.x; v < x.n; v += blockDim.x) g += (x.rp[v + 1] - x.rp[v] + 3) / 4;
    atomicAdd(&groups, g);
    SmallTile *tiles0 = (SmallTile *)(b + O_TILES0);
    for (int t = threadIdx.x; t < x.n_stiles; t += blockDim.x) {
        SmallTile tl{};
        tl.comp = t % NA_COPIES;
        tl.src0 = x.stile * t;
        tl.ns = min(x.stile, x.n_src - x.stile * t);
        tiles0[t] = tl;
    }
    const int32_t *reach = x.reach ? x.reach : zero;
    for (int v = threadIdx.x; v < x.n; v += blockDim.x) zero[v] = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < x.n_src; i += blockDim.x) {
        const int s = x.srcs ? x.srcs[i] : i;
        if (s < 0 || s >= x.n) {
            bad = 1;  // (any thread; all write the same value)
            srcs[i] = 0;
            ws[i] = 0.0;
            continue;
        }
        srcs[i] = s;
        ws[i] = (double)reach[s] + 1.0;
    }
    for (int t = threadIdx.x; t < x.n_tiles; t += blockDim.x) {
        SmallTile tl{};
        tl.comp = 0;
        tl.src0 = 64 * t;
        tl.ns = min(64, x.n_src - 64 * t);
        tiles[t] = tl;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        SmallComp c{};
        c.n = x.n;
        c.rp = x.rp;
        c.col = x.col;
        c.reach = reach;
        c.bc = x.bc;
        *(SmallComp *)(b + O_COMP) = c;
        for (int k = 0; k < NA_COPIES; ++k) {
            c.bc = bc0 + k * NA_N;
            ((SmallComp *)(b + O_COMP0))[k] = c;
        }
        for (int k = 0; k < 16; ++k) ctr[k] = 0;
        // (the LDS of the launch was sized from the caller's arc count)
        const bool fits = x.lds > 0 && src_waves(x.n, groups, x.lds) >= x.min_waves;
        ctr[N0] = !bad && fits ? x.n_stiles : 0;
        ctr[N1] = bad ? 0 : x.n_tiles;
        ctr[BAD] = bad;
    }
}

// After k_src: its BC joins the caller's unless a count overflowed.
__global__ __launch_bounds__(256) void k_na_add(unsigned char *b, double *bc, int n) {
    const int32_t *ctr = (const int32_t *)(b + O_CTR);
    if (ctr[N0] == 0 || ctr[C0 + 1] != 0) return;
    const double *bc0 = (const double *)(b + O_BC);
    const int v = blockIdx.x * 256 + threadIdx.x;
    if (v >= n) return;
    ExactSum sum;
#pragma unroll
    for (int k = 0; k < NA_COPIES; ++k) sum.add(bc0[k * NA_N + v]);
    if (sum.value() != 0.0) bc[v] += sum.value();
}

// The first pass listed the tiles whose 64-bit counts overflowed: they make
// the second pass's table.
__global__ __launch_bounds__(64) void k_na_remap(unsigned char *b) {
    int32_t *ctr = (int32_t *)(b + O_CTR);
    const SmallTile *t1 = (const SmallTile *)(b + O_TILES1);
    SmallTile *t2 = (SmallTile *)(b + O_TILES2);
    const int32_t *redo = (const int32_t *)(b + O_REDO1);
    const int k = ctr[C1 + 1];
    for (int i = threadIdx.x; i < k; i += blockDim.x) t2[i] = t1[redo[i]];
    if (threadIdx.x == 0) ctr[N2] = k;
}

static SmallArgs pass_args(unsigned char *b, bool second, int32_t n) {
    SmallArgs a{};
    a.comps = (const SmallComp *)(b + O_COMP);
    a.tiles = (const SmallTile *)(b + (second ? O_TILES2 : O_TILES1));
    a.n_tiles = 0;
    a.n_tiles_dev = (const int32_t *)(b + O_CTR) + (second ? N2 : N1);
    a.srcs = (const int32_t *)(b + O_SRCS);
    a.ws = (const double *)(b + O_WS);
    a.counter = (int32_t *)(b + O_CTR) + (second ? C2 : C1);
    a.redo = (int32_t *)(b + (second ? O_REDO2 : O_REDO1));
    a.sig = (uint64_t *)(b + O_SIG);
    a.tt = b + O_TT;
    a.Q = (int32_t *)(b + O_Q);
    a.Qm = (uint64_t *)(b + O_QM);
    a.slab = (int64_t)NA_SLAB;
    a.limit = 0;
    a.nmax = n;  // sizes the kernel's LDS
    return a;
}

extern "C" int bcx_bc_small_noalloc(bcx_ctx *ctx, int32_t n, int64_t arcs, const int32_t *d_row_ptr,
                                    const int32_t *d_col, const int32_t *d_reach, const int32_t *d_srcs,
                                    int32_t n_src, int32_t precision, double *d_bc) {
    if (!ctx) return BCX_E_ARG;
    if (n < 1 || n > NA_N)
        return ctx_fail(ctx, BCX_E_ARG, "bcx_bc_small_noalloc: n must be 1.." + std::to_string(NA_N) +
                                            " (BCX_NOALLOC_MAX_N), got " + std::to_string(n));
    if (!d_srcs) n_src = n;
    if (n_src < 1 || n_src > n) return ctx_fail(ctx, BCX_E_ARG, "bcx_bc_small_noalloc: n_src must be 1..n");
    if (arcs < 0 || (arcs > 0 && !d_col) || !d_row_ptr || !d_bc ||
        (precision != BCX_PREC_FP64 && precision != BCX_PREC_FP32C))
        return ctx_fail(ctx, BCX_E_ARG, "bcx_bc_small_noalloc: bad arguments");
    const int dev = ctx->device;
    unsigned char *base = nullptr;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        if (dev >= 0 && dev < 64) base = (unsigned char *)g_ptr[dev];
        if (!base)
            return ctx_fail(ctx, BCX_E_HIP, std::string("bcx_bc_small_noalloc: scratch array not available: ") +
                                                hipGetErrorString(dev >= 0 && dev < 64 ? g_err[dev] : hipErrorInvalidDevice));
    }
    int rc = ctx_hip(ctx, hipSetDevice(dev), "set device");
    if (rc) return rc;
    NaArgs x{};
    x.n = n;
    x.n_src = n_src;
    x.n_tiles = (n_src + 63) / 64;
    x.stile = n_src <= 4 * NA_STILES ? 4 : 8;
    x.n_stiles = (n_src + x.stile - 1) / x.stile;
    x.rp = d_row_ptr;
    x.col = d_col;
    x.reach = d_reach;
    x.srcs = d_srcs;
    x.bc = d_bc;
    x.base = base;
    const int grid = std::min(NA_WG, x.n_tiles);
    const bool fp32 = precision == BCX_PREC_FP32C;
    // rows of a arcs make at most a / 4 + n groups; a tile keeps stile sources
    // in flight, so two waves (three with FP32 terms) are where bcx_run draws
    // the line as well
    x.min_waves = fp32 ? 3 : 2;
    const int64_t lds = src_shared_bytes(n, arcs / 4 + n) + x.stile * src_wave_bytes(n);
    x.lds = (int32_t)std::min(SRC_LDS, lds);
    hipStream_t st = ctx->stream;
    int32_t status[16];
    auto read_status = [&]() {
        int r = ctx_hip(ctx, hipMemcpyAsync(status, base + O_CTR, sizeof(status), hipMemcpyDeviceToHost, st),
                        "no-alloc status");
        return r ? r : ctx_hip(ctx, hipStreamSynchronize(st), "no-alloc run");
    };
    hipLaunchKernelGGL(k_na_setup, dim3(1 + NA_COPIES), dim3(256), 0, st, x);
    if ((rc = ctx_hip(ctx, hipGetLastError(), "no-alloc setup"))) return rc;
    SrcArgs sa{};
    sa.comps = (const SmallComp *)(base + O_COMP0);
    sa.tiles = (const SmallTile *)(base + O_TILES0);
    sa.n_tiles_dev = (const int32_t *)(base + O_CTR) + N0;
    sa.lds = x.lds;
    sa.srcs = (const int32_t *)(base + O_SRCS);
    sa.ws = (const double *)(base + O_WS);
    sa.counter = (int32_t *)(base + O_CTR) + C0;
    sa.redo = (int32_t *)(base + O_REDO0);
    sa.stop = 1;
    if ((rc = ctx_hip(ctx, launch_src(sa, false, fp32, x.n_stiles, st), "no-alloc pass"))) return rc;
    hipLaunchKernelGGL(k_na_add, dim3((n + 255) / 256), dim3(256), 0, st, base, d_bc, n);
    if ((rc = ctx_hip(ctx, hipGetLastError(), "no-alloc add")) || (rc = read_status())) return rc;
    if (!status[BAD] && (status[N0] == 0 || status[C0 + 1] != 0)) {
        if ((rc = ctx_hip(ctx, launch_small(pass_args(base, false, n), false, fp32, grid, st), "no-alloc pass")))
            return rc;
        hipLaunchKernelGGL(k_na_remap, dim3(1), dim3(64), 0, st, base);
        if ((rc = ctx_hip(ctx, hipGetLastError(), "no-alloc remap")) ||
            (rc = ctx_hip(ctx, launch_small(pass_args(base, true, n), true, fp32, grid, st), "no-alloc FP64 pass")) ||
            (rc = read_status()))
            return rc;
    }
    if (status[BAD]) return ctx_fail(ctx, BCX_E_ARG, "bcx_bc_small_noalloc: a source is out of range");
    return BCX_OK;
}
