// Small components, one wave per source: the whole per-source state lives in
// LDS and a source runs from its first to its last level without a barrier.
//
// A workgroup takes a tile (component, up to 64 sources) from a work counter,
// copies the component's CSR into LDS, and its waves take the tile's sources
// one at a time.  Per source: a 2-bit level code per vertex (0: not reached,
// else 1 + level mod 3, which tells a neighbour's level exactly because an arc
// joins levels that differ by at most one), one 8-byte word per vertex and the
// list of vertices in level order, the first of each level flagged.
//
// Forward, one walk over the arcs of each level's vertices: arcs to the level
// below add its path count (exact uint64, FP64 in CSR order on overflow), arcs
// to unreached vertices append them to the list.  Backward, one walk: rho_v =
// sum over successors of t_w, t_v = (r(v)+1)/sigma_v + rho_v, which takes the
// place of sigma_v in the vertex's word (the predecessors need t_v alone);
// FP32 terms with Kahan compensation or FP64, summed in CSR order.  The BC of
// a tile is accumulated in LDS and added to the component once per tile.
// (Codes/kernels_free.cu:154-473 computes the same, one source per block with
// its state in global memory.)
//
// What bounds it: the round trips to LDS of a wave's arc steps (four arcs of
// each lane's row at a time) and LDS gathers; no step waits for another wave or
// for global memory.  Measured against 64 sources per wave with rows in global
// memory and barriers per level (bcx_small.hip; 10k-vertex workload of 16
// blocks, all sources, one launch): 0.28 ms FP64 and 0.36 ms FP32C against
// 0.81 ms, and against one source per workgroup with endpoint rows
// (bcx_plain.hip, 48 launches): 10.1 ms to 0.31 ms for the whole run.
//
// A tile in which a uint64 count overflows adds nothing and is listed for an
// FP64 rerun, as in the 64-source kernel (bcx_small.hip).
#include "bcx_src.h"
#include "bcx_device.h"

namespace bcx {

namespace {

constexpr int XB = 64 * SRC_WAVES;  // threads of a workgroup
// Rows longer than this are walked by the whole wave, shorter ones by a lane.
constexpr int XROW = 64;
constexpr uint16_t FIRST = 0x8000;  // list flag: first vertex of its level

__device__ __forceinline__ uint64_t xl64(uint64_t x, int src) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, src);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(x >> 32), src);
    return ((uint64_t)hi << 32) | lo;
}

// Orders the wave's own LDS accesses (executed in order) for the compiler.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

struct KahanX {
    float s = 0.f, c = 0.f;
    __device__ __forceinline__ void add(float x) {
        const float y = x - c;
        const float t = s + y;
        c = (t - s) - y;
        s = t;
    }
    __device__ __forceinline__ double value() const { return (double)s - (double)c; }
};
struct SumX {
    double s = 0.0;
    __device__ __forceinline__ void add(double x) { s += x; }
    __device__ __forceinline__ double value() const { return s; }
};
// path-count sums: exact uint64 with a wrap flag, or FP64
template <bool F64>
struct SigX {
    uint64_t u = 0;
    double d = 0.0;
    bool wrap = false;
    __device__ __forceinline__ void add(uint64_t x) {
        if (F64) {
            d += u2d(x);
        } else {
            const uint64_t s = u + x;
            wrap |= s < u;
            u = s;
        }
    }
    __device__ __forceinline__ uint64_t bits() const { return F64 ? d2u(d) : u; }
};

struct WaveState {
    uint64_t *st;   // [n] path count, then term
    uint32_t *lv;   // [(n + 15) / 16] level codes, 16 per word
    uint16_t *S;    // [n] vertices in level order
};

template <typename TT>
__device__ __forceinline__ TT term(const uint64_t *st, int w) {
    return *(const TT *)&st[w];
}

// One source.  Returns false when a uint64 count overflowed (nothing added).
template <bool F64, typename TT>
__device__ __forceinline__ bool src_run(const SrcArgs &a, int n, int s, double ws, const int32_t *rp,
                                        const uint16_t *col, const gint *reach, double *bc, const WaveState &x,
                                        int slot, int *depth) {
    using Acc = typename std::conditional<sizeof(TT) == 4, KahanX, SumX>::type;
    const int lane = threadIdx.x & 63;
    const uint64_t below = (1ull << lane) - 1;
    uint64_t *st = x.st;
    uint32_t *lv = x.lv;
    uint16_t *S = x.S;
    for (int i = lane; i < (n + 15) / 16; i += 64) lv[i] = 0;
    wave_sync();
    if (lane == 0) {
        lv[s >> 4] = 1u << (2 * (s & 15));
        S[0] = (uint16_t)s | FIRST;
        st[s] = F64 ? d2u(1.0) : 1ull;
    }
    wave_sync();
    // ----------------------------------------------------------- forward
    int q0 = 0, q1 = 1, l = 0;
    uint32_t cprev = 3, cnext = 2;  // codes of levels l-1 (l = 0: none set) and l+1
    bool ovf = false;
    while (true) {
        int tail = q1;  // wave-uniform
        for (int base = q0; base < q1; base += 64) {
            const int e = base + lane;
            int v = 0, j0 = 0, j1 = 0;
            if (e < q1) {
                v = S[e] & ~FIRST;
                j0 = rp[v];
                j1 = rp[v + 1];
            }
            const uint64_t wide = __ballot(j1 - j0 > XROW);
            const int je = j1 - j0 > XROW ? j0 : j1;
            SigX<F64> acc;
            // the lanes' rows, four arcs of each at a time
            for (int j = j0; __ballot(j < je); j += 4) {
                int w[4];
                uint32_t f[4];
                uint64_t y[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) w[u] = j + u < je ? col[j + u] : -1;
#pragma unroll
                for (int u = 0; u < 4; ++u) f[u] = w[u] >= 0 ? (lv[w[u] >> 4] >> (2 * (w[u] & 15))) & 3u : cnext;
#pragma unroll
                for (int u = 0; u < 4; ++u) y[u] = f[u] == cprev ? st[w[u]] : 0;
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (f[u] == cprev) acc.add(y[u]);
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    bool mine = false;
                    if (f[u] == 0) {
                        const int sh = 2 * (w[u] & 15);
                        const uint32_t old = atomicOr(&lv[w[u] >> 4], cnext << sh);
                        mine = ((old >> sh) & 3u) == 0;
                    }
                    const uint64_t b = __ballot(mine);
                    if (mine) {
                        const int pos = tail + __popcll(b & below);
                        S[pos] = (uint16_t)w[u] | (pos == q1 ? FIRST : 0);
                    }
                    tail += __popcll(b);
                }
            }
            // long rows: the wave walks one at a time, its counts summed in CSR order
            for (uint64_t m = wide; m; m &= m - 1) {
                const int src = __ffsll((long long)m) - 1;
                const int a0 = __builtin_amdgcn_readlane(j0, src), a1 = __builtin_amdgcn_readlane(j1, src);
                SigX<F64> sum;
                for (int c = a0; c < a1; c += 64) {
                    const int w = c + lane < a1 ? col[c + lane] : -1;
                    const uint32_t f = w >= 0 ? (lv[w >> 4] >> (2 * (w & 15))) & 3u : cnext;
                    const uint64_t y = f == cprev ? st[w] : 0;
                    for (uint64_t r = __ballot(f == cprev); r; r &= r - 1) sum.add(xl64(y, __ffsll((long long)r) - 1));
                    bool mine = false;
                    if (f == 0) {
                        const int sh = 2 * (w & 15);
                        const uint32_t old = atomicOr(&lv[w >> 4], cnext << sh);
                        mine = ((old >> sh) & 3u) == 0;
                    }
                    const uint64_t b = __ballot(mine);
                    if (mine) {
                        const int pos = tail + __popcll(b & below);
                        S[pos] = (uint16_t)w | (pos == q1 ? FIRST : 0);
                    }
                    tail += __popcll(b);
                }
                if (lane == src) acc = sum;
            }
            if (e < q1) {
                if (l > 0) {
                    st[v] = acc.bits();
                    if (!F64) ovf |= acc.wrap || (a.limit && acc.u >= a.limit);
                }
                if (a.lvl) a.lvl[(int64_t)v * 64 + slot] = l;
                if (a.psig) a.psig[(int64_t)v * 64 + slot] = l > 0 ? acc.bits() : (F64 ? d2u(1.0) : 1ull);
            }
        }
        wave_sync();
        if (!F64 && __ballot(ovf)) return false;
        if (tail == q1) break;
        q0 = q1;
        q1 = tail;
        l++;
        const uint32_t c = cprev;  // l-1 <- l, l+1 <- l+2, whose code is the old l-1's
        cprev = 6 - cprev - cnext;
        cnext = c;
    }
    if (lane == 0) atomicMax(depth, l);
    // ---------------------------------------------------------- backward
    // [q0, q1) is the deepest level l; code of level l: 1 + l % 3
    int b1 = q1;
    for (int d = l; d >= 1; --d) {
        // the first vertex of the level: the last flag below b1
        int b0 = b1;
        while (true) {
            const int e = b0 - 64 + lane;
            const uint64_t fl = __ballot(e >= 0 && (S[e < 0 ? 0 : e] & FIRST));
            if (fl) {
                b0 = b0 - 64 + (63 - __clzll((long long)fl));
                break;
            }
            b0 -= 64;
        }
        const uint32_t csucc = 1 + (uint32_t)((d + 1) % 3);
        for (int base = b0; base < b1; base += 64) {
            const int e = base + lane;
            int v = 0, j0 = 0, j1 = 0, rv = 0;
            uint64_t sx = 0;
            if (e < b1) {
                v = S[e] & ~FIRST;
                j0 = rp[v];
                j1 = rp[v + 1];
                rv = reach[v];
                sx = st[v];
            }
            Acc acc;
            if (d < l) {
                const uint64_t wide = __ballot(j1 - j0 > XROW);
                const int je = j1 - j0 > XROW ? j0 : j1;
                for (int j = j0; __ballot(j < je); j += 4) {
                    int w[4];
                    bool use[4];
                    TT t[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) w[u] = j + u < je ? col[j + u] : -1;
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        use[u] = w[u] >= 0 && ((lv[w[u] >> 4] >> (2 * (w[u] & 15))) & 3u) == csucc;
#pragma unroll
                    for (int u = 0; u < 4; ++u) t[u] = use[u] ? term<TT>(st, w[u]) : (TT)0;
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        if (use[u]) acc.add(t[u]);
                }
                for (uint64_t m = wide; m; m &= m - 1) {
                    const int src = __ffsll((long long)m) - 1;
                    const int a0 = __builtin_amdgcn_readlane(j0, src), a1 = __builtin_amdgcn_readlane(j1, src);
                    Acc sum;
                    for (int c = a0; c < a1; c += 64) {
                        const int w = c + lane < a1 ? col[c + lane] : -1;
                        const bool use = w >= 0 && ((lv[w >> 4] >> (2 * (w & 15))) & 3u) == csucc;
                        const double t = use ? (double)term<TT>(st, w) : 0.0;
                        for (uint64_t r = __ballot(use); r; r &= r - 1)
                            sum.add((TT)u2d(xl64(d2u(t), __ffsll((long long)r) - 1)));
                    }
                    if (lane == src) acc = sum;
                }
            }
            if (e < b1) {
                const double sv = F64 ? u2d(sx) : (double)sx;
                const double rho = acc.value();
                const double delta = sv * rho;
                *(TT *)&st[v] = (TT)(((double)rv + 1.0) / sv + rho);
                if (delta != 0.0) unsafeAtomicAdd(&bc[v], ws * delta);
                if (a.dbg) a.dbg[(int64_t)v * 64 + slot] = delta;
            }
        }
        wave_sync();
        b1 = b0;
    }
    return true;
}

}  // namespace

template <bool F64, typename TT>
__global__ __launch_bounds__(XB) void k_src(SrcArgs a) {
    extern __shared__ __align__(16) unsigned char s_lds[];
    __shared__ int s_item, s_next, s_ovf, s_depth;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int n_tiles = a.n_tiles_dev ? *a.n_tiles_dev : a.n_tiles;
    while (true) {
        if (tid == 0) {
            s_item = atomicAdd(&a.counter[0], 1);
            s_next = 0;
            s_ovf = 0;
            s_depth = 0;
        }
        __syncthreads();
        const int item = s_item;
        if (item >= n_tiles) break;
        const SmallTile tl = a.tiles[item];
        const SmallComp cp = a.comps[tl.comp];
        const int n = cp.n;
        const gint *grp = glb(cp.rp), *gcol = glb(cp.col), *reach = glb(cp.reach);
        const int r0 = grp[0], m = grp[n] - r0;
        double *bc = (double *)s_lds;
        int32_t *rp = (int32_t *)(s_lds + src_up16(8 * (int64_t)n));
        uint16_t *col = (uint16_t *)((unsigned char *)rp + src_up16(4 * ((int64_t)n + 1)));
        const int64_t wb = src_wave_bytes(n);
        const int waves = (int)src_waves(n, m, a.lds);
        for (int v = tid; v < n; v += XB) bc[v] = 0.0;
        for (int v = tid; v <= n; v += XB) rp[v] = grp[v] - r0;
        for (int j = tid; j < m; j += XB) col[j] = (uint16_t)gcol[r0 + j];
        __syncthreads();
        if (wv < waves) {
            unsigned char *p = s_lds + src_shared_bytes(n, m) + wv * wb;
            WaveState x;
            x.st = (uint64_t *)p;
            x.lv = (uint32_t *)(p + src_up16(8 * (int64_t)n));
            x.S = (uint16_t *)((unsigned char *)x.lv + src_up16(4 * (((int64_t)n + 15) / 16)));
            while (true) {
                int i = 0;
                if (lane == 0) i = atomicAdd(&s_next, 1);
                i = __builtin_amdgcn_readlane(i, 0);
                if (i >= tl.ns) break;
                const int s = __builtin_amdgcn_readfirstlane(a.srcs[tl.src0 + i]);
                if (!src_run<F64, TT>(a, n, s, a.ws[tl.src0 + i], rp, col, reach, bc, x, i,
                                         &s_depth)) {
                    if (lane == 0) s_ovf = 1;
                    break;
                }
            }
        }
        __syncthreads();
        if (s_ovf) {
            if (tid == 0) a.redo[atomicAdd(&a.counter[1], 1)] = item;
        } else {
            if (tid == 0) atomicMax(&a.counter[2], s_depth);
            for (int v = tid; v < n; v += XB)
                if (bc[v] != 0.0) gadd(glb(cp.bc) + v, bc[v]);
        }
        __syncthreads();
    }
}

// FP64-sigma tiles keep FP64 terms in either precision: 1/sigma can leave
// the f32 range.
hipError_t launch_src(const SrcArgs &a, bool f64, bool fp32, int grid, hipStream_t st) {
    if (a.lds < 0 || a.lds > SRC_LDS) return hipErrorInvalidValue;
    if (f64) hipLaunchKernelGGL((k_src<true, double>), dim3(grid), dim3(XB), a.lds, st, a);
    else if (fp32) hipLaunchKernelGGL((k_src<false, float>), dim3(grid), dim3(XB), a.lds, st, a);
    else hipLaunchKernelGGL((k_src<false, double>), dim3(grid), dim3(XB), a.lds, st, a);
    return hipGetLastError();
}

int src_blocks_per_cu(int lds) {
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, (const void *)&k_src<false, float>, XB, lds) != hipSuccess ||
        nb < 1) {
        (void)hipGetLastError();
        nb = 1;
    }
    return nb;
}

}  // namespace bcx
