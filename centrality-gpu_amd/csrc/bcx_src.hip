// Small components, one wave per source: the whole per-source state lives in
// LDS and a source runs from its first to its last level without a barrier.
//
// A workgroup takes a tile (component, up to 64 sources) from a work counter,
// copies the component's CSR into LDS, and its waves take the tile's sources
// one at a time.  Per source: a level code per vertex (0: not reached, else
// 1 + level mod 3, which tells a neighbour's level exactly because an arc joins
// levels that differ by at most one), one 8-byte word per vertex and the list
// of vertices in level order, the first of each level flagged.
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
// What bounds it: vector issue (61% of a busy compute unit's cycles with FP64
// terms, 63% with FP32 ones) and the LDS round trips of a wave's arc steps; no
// step waits for another wave or for global memory.  A step takes a group of four arcs of each lane's row (rows are
// padded to whole groups, so no arc is tested for the row's end) and is free of
// branches, so its accesses are in flight together.  Measured, 10k-vertex
// workload of 16 blocks, all sources, whole run: 0.25 ms FP64 and 0.28 ms FP32C
// (0.31 and 0.40 ms with single-arc bounds tests, 2-bit codes set by LDS
// atomics and 64-source tiles), against 0.86 ms with 64 sources per wave, rows in
// global memory and barriers per level (bcx_small.hip) and 10.1 ms with one
// source per workgroup and endpoint rows (bcx_plain.hip, 48 launches).
//
// A tile in which a uint64 count overflows adds nothing and is listed for an
// FP64 rerun, as in the 64-source kernel (bcx_small.hip).
#include "bcx_src.h"
#include "bcx_device.h"

namespace bcx {

namespace {

constexpr int XB = 64 * SRC_WAVES;  // threads of a workgroup
// Rows of more groups than this are walked by the whole wave, shorter ones by a
// lane, a group of four arcs per step.
constexpr int XROW = 16;
constexpr uint16_t FIRST = 0x8000;  // list flag: first vertex of its level

__device__ __forceinline__ uint64_t xl64(uint64_t x, int src) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, src);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(x >> 32), src);
    return ((uint64_t)hi << 32) | lo;
}

// ballot of a predicate, and the number of its lanes below this one
__device__ __forceinline__ uint64_t bal(bool p) { return __builtin_amdgcn_ballot_w64(p); }
__device__ __forceinline__ int rank_in(uint64_t b, int from) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, (uint32_t)from));
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
            wrap |= __builtin_add_overflow(u, x, &u);
        }
    }
    __device__ __forceinline__ uint64_t bits() const { return F64 ? d2u(d) : u; }
};

// A wave's state; entries n and n + 1 of each array belong to no vertex: a lane
// without an arc reads n (word 0, a code that matches none) and one with nothing
// to store writes n + 1, so the arc steps have no branches and their LDS
// accesses are in flight together.
struct WaveState {
    uint64_t *st;   // [n + 2] path count, then term
    uint8_t *lv;    // [n + 2] level codes
    uint16_t *S;    // [n + 2] vertices in level order
};
constexpr uint32_t NO_LEVEL = 4;  // lv[n]
constexpr uint32_t REACHED = 8;   // reached by the level being walked, not yet listed

// The vertices of arc group g (group `none` holds no arcs: every entry is n).
__device__ __forceinline__ void arcs4(const uint64_t *col, int g, int (&w)[4]) {
    const uint64_t x = col[g];
    w[0] = (int)((uint32_t)x & 0xffffu);
    w[1] = (int)((uint32_t)x >> 16);
    w[2] = (int)((uint32_t)(x >> 32) & 0xffffu);
    w[3] = (int)((uint32_t)(x >> 48));
}

// Lists the vertices marked REACHED in id order (four per lane and step) and
// gives them the code of the next level; returns the list's end.
__device__ __forceinline__ int list_reached(const WaveState &x, int n, uint32_t cnext, int q1) {
    const int lane = threadIdx.x & 63;
    uint32_t *lv4 = (uint32_t *)x.lv;
    int tail = q1;
    for (int i = lane; i - lane < (n + 3) / 4; i += 64) {
        const uint32_t c = 4 * i < n ? lv4[i] : 0;
        const uint32_t m = c & (REACHED * 0x01010101u);
        if (!bal(m != 0)) continue;
        if (m) lv4[i] = (c ^ m) | (m / REACHED) * cnext;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const bool mine = (m >> (8 * k)) & REACHED;
            const uint64_t b = bal(mine);
            if (mine) {
                const int pos = rank_in(b, tail);
                x.S[pos] = (uint16_t)(4 * i + k) | (pos == q1 ? FIRST : 0);
            }
            tail += __popcll(b);
        }
    }
    return tail;
}

template <typename TT>
__device__ __forceinline__ TT term(const uint64_t *st, int w) {
    return *(const TT *)&st[w];
}

// Appends the vertices w of the lanes that found code 0 to the list (once
// each: of the lanes that write their mark into a vertex's unused word, the one
// that reads it back appends) and gives them the code of the next level.
// Returns the list's end.
template <int U>
__device__ __forceinline__ int discover(const WaveState &x, int n, const int (&w)[U], const uint32_t (&f)[U],
                                        uint32_t cnext, int q1, int tail) {
    const int lane = threadIdx.x & 63;
    bool any = false;
#pragma unroll
    for (int u = 0; u < U; ++u) any |= f[u] == 0;
    if (!bal(any)) return tail;
    int at[U];
    uint32_t got[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        at[u] = f[u] == 0 ? w[u] : n + 1;
        *(uint32_t *)&x.st[at[u]] = (uint32_t)(64 * u + lane);
    }
    wave_sync();
#pragma unroll
    for (int u = 0; u < U; ++u) got[u] = *(const uint32_t *)&x.st[at[u]];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        x.lv[at[u]] = (uint8_t)cnext;
        const bool mine = f[u] == 0 && got[u] == (uint32_t)(64 * u + lane);
        const uint64_t b = bal(mine);
        const int pos = rank_in(b, tail);
        x.S[mine ? pos : n + 1] = (uint16_t)(w[u] | (pos == q1 ? FIRST : 0));
        tail += __popcll(b);
    }
    return tail;
}

// One source.  Returns false when a uint64 count overflowed (nothing added).
template <bool F64, typename TT>
__device__ __forceinline__ bool src_run(const SrcArgs &a, int n, int s, double ws, const int32_t *rp,
                                        const uint64_t *col, const gint *reach, double *bc, const WaveState &x,
                                        int slot, int *depth) {
    using Acc = typename std::conditional<sizeof(TT) == 4, KahanX, SumX>::type;
    const int lane = threadIdx.x & 63;
    uint64_t *st = x.st;
    uint8_t *lv = x.lv;
    uint16_t *S = x.S;
    for (int i = lane; i < (n + 2 + 3) / 4; i += 64) ((uint32_t *)lv)[i] = 0;
    wave_sync();
    if (lane == 0) {
        lv[n] = NO_LEVEL;
        lv[s] = 1;
        S[0] = (uint16_t)s | FIRST;
        st[n] = 0;
        st[s] = F64 ? d2u(1.0) : 1ull;
    }
    wave_sync();
    // ----------------------------------------------------------- forward
    int q0 = 0, q1 = 1, l = 0;
    uint32_t cprev = 3, cnext = 2;  // codes of levels l-1 (l = 0: none set) and l+1
    bool ovf = false;
    const int none = rp[n];
    while (true) {
        int tail = q1;  // wave-uniform
        // a wide level marks what it reaches and lists it by one pass over the
        // codes, a narrow one lists as it goes (a pass costs about 45
        // instructions per 256 vertices, listing about 75 per arc step)
        const bool marks = 16 * (q1 - q0) > n;
        for (int base = q0; base < q1; base += 64) {
            const int e = base + lane;
            int v = 0, j0 = 0, j1 = 0;
            if (e < q1) {
                v = S[e] & ~FIRST;
                j0 = rp[v];
                j1 = rp[v + 1];
            }
            const uint64_t wide = bal(j1 - j0 > XROW);
            const int je = j1 - j0 > XROW ? j0 : j1;
            SigX<F64> acc;
            for (int j = j0; bal(j < je); ++j) {
                int w[4];
                uint32_t f[4];
                uint64_t y[4];
                arcs4(col, j < je ? j : none, w);
#pragma unroll
                for (int u = 0; u < 4; ++u) f[u] = lv[w[u]];
#pragma unroll
                for (int u = 0; u < 4; ++u) y[u] = st[f[u] == cprev ? w[u] : n];
#pragma unroll
                for (int u = 0; u < 4; ++u) acc.add(y[u]);
                if (marks) {
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        if (f[u] == 0) lv[w[u]] = (uint8_t)REACHED;
                } else {
                    tail = discover<4>(x, n, w, f, cnext, q1, tail);
                }
                wave_sync();
            }
            // long rows: the wave walks one at a time, its counts summed in CSR order
            for (uint64_t m = wide; m; m &= m - 1) {
                const int src = __ffsll((long long)m) - 1;
                const int a0 = __builtin_amdgcn_readlane(j0, src), a1 = __builtin_amdgcn_readlane(j1, src);
                SigX<F64> sum;
                for (int c = 4 * a0; c < 4 * a1; c += 64) {
                    int w[1];
                    uint32_t f[1];
                    w[0] = c + lane < 4 * a1 ? ((const uint16_t *)col)[c + lane] : n;
                    f[0] = lv[w[0]];
                    const uint64_t y = st[f[0] == cprev ? w[0] : n];
                    for (uint64_t r = bal(f[0] == cprev); r; r &= r - 1)
                        sum.add(xl64(y, __ffsll((long long)r) - 1));
                    if (marks) {
                        if (f[0] == 0) lv[w[0]] = (uint8_t)REACHED;
                    } else {
                        tail = discover<1>(x, n, w, f, cnext, q1, tail);
                    }
                    wave_sync();
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
        if (marks) {
            tail = list_reached(x, n, cnext, q1);
            wave_sync();
        }
        if (!F64 && bal(ovf)) return false;
        if (tail == q1) break;
        q0 = q1;
        q1 = __builtin_amdgcn_readfirstlane(tail);
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
            const uint64_t fl = bal(e >= 0 && (S[e < 0 ? 0 : e] & FIRST));
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
                rv = reach[v];
                j0 = rp[v];
                j1 = rp[v + 1];
                sx = st[v];
            }
            Acc acc;
            if (d < l) {
                const uint64_t wide = bal(j1 - j0 > XROW);
                const int je = j1 - j0 > XROW ? j0 : j1;
                for (int j = j0; bal(j < je); ++j) {
                    int w[4];
                    bool use[4];
                    TT t[4];
                    arcs4(col, j < je ? j : none, w);
#pragma unroll
                    for (int u = 0; u < 4; ++u) use[u] = lv[w[u]] == csucc;
#pragma unroll
                    for (int u = 0; u < 4; ++u) t[u] = term<TT>(st, use[u] ? w[u] : n);
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        // (adding the empty word's 0 leaves an FP64 sum as it
                        // is, not a compensated one)
                        Acc more = acc;
                        more.add(t[u]);
                        if (sizeof(TT) == 8 || use[u]) acc = more;
                    }
                }
                for (uint64_t m = wide; m; m &= m - 1) {
                    const int src = __ffsll((long long)m) - 1;
                    const int a0 = __builtin_amdgcn_readlane(j0, src), a1 = __builtin_amdgcn_readlane(j1, src);
                    Acc sum;
                    for (int c = 4 * a0; c < 4 * a1; c += 64) {
                        const int w = c + lane < 4 * a1 ? ((const uint16_t *)col)[c + lane] : n;
                        const bool use = lv[w] == csucc;
                        const double t = (double)term<TT>(st, use ? w : n);
                        for (uint64_t r = bal(use); r; r &= r - 1)
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
    __shared__ int s_item, s_next, s_ovf, s_depth, s_scan[SRC_WAVES];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int n_tiles = a.n_tiles_dev ? *a.n_tiles_dev : a.n_tiles;
    // the first tile is the workgroup's own, the work counter hands out the rest
    for (bool first = true;; first = false) {
        if (tid == 0) {
            if (a.stop && ald(&a.counter[1]) != 0) s_item = n_tiles;
            else if (first) s_item = blockIdx.x;
            else s_item = (int)gridDim.x < n_tiles ? (int)gridDim.x + atomicAdd(&a.counter[0], 1) : n_tiles;
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
        double *bc = (double *)s_lds;
        int32_t *rp = (int32_t *)(s_lds + src_up16(8 * (int64_t)n));
        uint64_t *col = (uint64_t *)((unsigned char *)rp + src_up16(4 * ((int64_t)n + 1)));
        // row pointers in groups of four arcs: a scan of the padded rows, XB at
        // a time
        int groups = 0;
        for (int base = 0; base < n; base += XB) {
            const int v = base + tid;
            const int d = v < n ? (grp[v + 1] - grp[v] + 3) / 4 : 0;
            int inc = d;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int y = __shfl_up(inc, o, 64);
                if (lane >= o) inc += y;
            }
            if (lane == 63) s_scan[wv] = inc;
            __syncthreads();
            int before = groups;
            for (int k = 0; k < SRC_WAVES; ++k) {
                before += k < wv ? s_scan[k] : 0;
                groups += s_scan[k];
            }
            if (v < n) rp[v] = before + inc - d;
            __syncthreads();
        }
        if (tid == 0) rp[n] = groups;
        const int64_t wb = src_wave_bytes(n);
        const int waves = (int)src_waves(n, groups, a.lds);
        const int accs = sizeof(TT) == 8 ? src_accs(n, groups, a.lds) : 1;
        double *more = (double *)(s_lds + src_shared_bytes(n, groups) + waves * wb);  // the accumulators past the first
        const int acc_words = (int)(src_up16(8 * (int64_t)n) / 8);
        for (int v = tid; v < n; v += XB) bc[v] = 0.0;
        for (int v = tid; v < (accs - 1) * acc_words; v += XB) more[v] = 0.0;
        for (int g = tid; g <= groups; g += XB) col[g] = 0x0001000100010001ull * (uint64_t)n;
        __syncthreads();
        for (int v = wv; v < n; v += SRC_WAVES) {  // (a wave per row)
            const int r0 = grp[v], d = grp[v + 1] - r0;
            for (int j = lane; j < d; j += 64) ((uint16_t *)col)[4 * rp[v] + j] = (uint16_t)gcol[r0 + j];
        }
        __syncthreads();
        if (wv < waves) {
            unsigned char *p = s_lds + src_shared_bytes(n, groups) + wv * wb;
            WaveState x;
            x.st = (uint64_t *)p;
            x.lv = p + src_up16(8 * ((int64_t)n + 2));
            x.S = (uint16_t *)(x.lv + src_up16((int64_t)n + 2));
            const int own = wv & (accs - 1);
            double *acc = own ? more + (own - 1) * acc_words : bc;
            while (true) {
                int i = 0;
                if (lane == 0) i = atomicAdd(&s_next, 1);
                i = __builtin_amdgcn_readlane(i, 0);
                if (i >= tl.ns) break;
                const int s = __builtin_amdgcn_readfirstlane(a.srcs[tl.src0 + i]);
                if (!src_run<F64, TT>(a, n, s, a.ws[tl.src0 + i], rp, col, reach, acc, x, i,
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
            gdbl *to = glb(cp.bc) + (item % SRC_COPIES) * a.copy;
            for (int v = tid; v < n; v += XB) {
                double sum = bc[v];
                if (accs == 2) sum += more[v];
                if (accs == 4) sum = (sum + more[v]) + (more[acc_words + v] + more[2 * acc_words + v]);
                if (sum != 0.0) gadd(to + v, sum);
            }
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

// Words that no tile added to are left alone: other components' runs may be adding
// to theirs.
__global__ __launch_bounds__(256) void k_src_fold(double *bc, int64_t copy, int64_t n, double *out, const int32_t *ctr,
                                                  int32_t *ctr_out) {
    const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (ctr && v < 3) ctr_out[v] = ctr[v];
    if (v >= n) return;
    double x[SRC_COPIES];
    bool any = false;
#pragma unroll
    for (int k = 0; k < SRC_COPIES; ++k) {
        x[k] = bc[v + k * copy];
        any |= k > 0 && x[k] != 0.0;
    }
    ExactSum s;
#pragma unroll
    for (int k = 0; k < SRC_COPIES; ++k) s.add(x[k]);
    if (any) {
#pragma unroll
        for (int k = 1; k < SRC_COPIES; ++k) bc[v + k * copy] = 0.0;
        ast((uint64_t *)&bc[v], d2u(s.value()));
    }
    if (out) out[v] = s.value();
}

hipError_t launch_src_fold(double *bc, int64_t copy, int64_t n, double *out, const int32_t *ctr, int32_t *ctr_out,
                           hipStream_t st) {
    hipLaunchKernelGGL(k_src_fold, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, bc, copy, n, out, ctr, ctr_out);
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
