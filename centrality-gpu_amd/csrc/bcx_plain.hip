// Plain per-source path: one workgroup per source, persistent grid with an
// atomic work counter (the schedule of Codes/kernels_free.cu:154-473 and
// Codes/kernels_active.cu:263-602), written for wave64 gfx950.
//
// A level code of two bits per vertex (0: not reached, else 1 + level mod 3) is
// all that an arc needs to know about its far end, because an arc joins levels
// that differ by at most one.  The codes of a source sit in LDS (n / 4 bytes),
// so an arc that leads nowhere costs no access to global memory.
//
// Forward, one walk over the arcs of each level's vertices: an arc to the level
// below adds its path count (exact uint64 with the wrap of any sum flagged; in
// FP64 mode the sum runs in CSR order, the oracle's, so FP64 counts are
// bit-exact), an arc to an unreached vertex takes it by an LDS atomic and
// appends it to the level-ordered list.  Backward, one walk: rho_v = sum of t_w
// over successors, t_v = (r(v)+1)/sigma_v + rho_v, delta_v = sigma_v rho_v
// (Codes/kernels_free.cu:378-421 computes the same with a division and three
// gathers per arc); BC[v] gets (r(s)+1) delta_v through FP64 atomics
// (Codes/kernels_free.cu:423-426).  t_v takes the place of sigma_v.
//
// What bounds it: the gathers of counts and terms along shortest-path arcs,
// whose lines miss L2 on cores of 10^5 vertices (12.7 us per source of an 84k
// core, the same with 256 and 512 sources in flight), and the dependent loads
// per level on deep graphs.  Against level words, list marks and count atomics
// in global memory with a lane per vertex: 1000 sources of the 84k core 165 ->
// 19 ms, 2049 sources of an 18.6k grid 27.4 -> 5.1 ms; with chain sources run
// directly, the core's BFS-ordered copy and dependencies added in vertex order
// 11.5 and 3.2 ms.
//
// A wave takes 64 vertices of a level.  Short rows are walked by a lane each,
// four arcs per step; longer ones as one flat range with a lane per arc, whose
// row is found by a search over the rows' first arcs in LDS and whose value is
// added to the row's sum in LDS; rows above HUB arcs by the whole wave.
//
// Chain sources: combine of two endpoint rows (Codes/postprocesses.cu:276-363)
// and level buckets by a counting sort in place of the CUB radix sort
// (Codes/postprocesses.cu:143-155), then the same backward.
#include "bcx_device.h"
#include "bcx_kernels.h"

#include <algorithm>

namespace bcx {

namespace {

constexpr int SHORT = 8;          // rows of a wave's vertices up to which a lane walks its own
constexpr int HUB = 256;          // degree above which a wave walks a row alone
constexpr int LDS_LEVELS = 1024;  // level offsets (chain kernel: level histogram) held in LDS
constexpr int PMAXW = 16;         // waves of a workgroup at most
// vertices whose level codes fit in LDS beside a workgroup's other arrays;
// above, the codes live in the workgroup's rows in global memory
constexpr int LV_LDS_N = 400000;

// LDS of one wave: the flat walk's first arcs, their offset into the CSR and
// the rows' sums
struct WaveRows {
    int P[64], A[64];
    uint64_t acc[64];
};
// with compensated FP32 terms, also a step's terms in arc order and the number
// of them before each arc
struct WaveTerms {
    float t[64 * 4 + 4];  // (read four at a time)
    uint16_t before[64 * 4 + 4];  // (the waves' parts stay 8-byte aligned)
};
// with FP64 terms, a row's sum in four parts, by lane: a part of a row of HUB arcs
// adds 64 terms one by one at most (100 sources of a 17k power-law core, error
// against 64 bits: one part 3.3e-16, four 1.4e-16, the same time)
struct WaveSums {
    double s[4 * 64];
};
template <typename TT>
__host__ __device__ constexpr int wave_lds() {
    return (int)(sizeof(WaveRows) + (sizeof(TT) == 4 ? sizeof(WaveTerms) : sizeof(WaveSums)));
}

struct KahanP {
    float s = 0.f, c = 0.f;
    __device__ __forceinline__ void add(float x) {
        const float y = x - c;
        const float t = s + y;
        c = (t - s) - y;
        s = t;
    }
    __device__ __forceinline__ double value() const { return (double)s - (double)c; }
};
struct SumP {
    double s = 0.0;
    __device__ __forceinline__ void add(double x) { s += x; }
    __device__ __forceinline__ double value() const { return s; }
};

struct PlainShared {
    int cnt[3];  // vertices appended at a level, by level mod 3
    int ovf[3];  // a count of the level overflowed, likewise
    int item, stop, top;
    int off[LDS_LEVELS];
};

__device__ __forceinline__ uint64_t sig_one(bool f64) { return f64 ? d2u(1.0) : 1ull; }
__device__ __forceinline__ uint64_t pbal(bool p) { return __builtin_amdgcn_ballot_w64(p); }
__device__ __forceinline__ int prank(uint64_t b, int from) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, (uint32_t)from));
}
__device__ __forceinline__ uint64_t prl64(uint64_t x, int src) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, src);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(x >> 32), src);
    return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ void psync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Workgroup barrier after every outstanding memory access of the wave.
__device__ __forceinline__ void pbarrier() {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
}

// Level codes, 16 per word, in LDS or (LG) in global memory, where they are
// set by L2 atomics and read past the vector L1.
template <bool LG>
struct Codes {
    uint32_t *w;
    __device__ __forceinline__ uint32_t get(int v) const {
        const uint32_t x = LG ? (uint32_t)ald((const int32_t *)&w[v >> 4]) : w[v >> 4];
        return (x >> (2 * (v & 15))) & 3u;
    }
    // sets an unset code; true for the one that did
    __device__ __forceinline__ bool take(int v, uint32_t c) const {
        const int sh = 2 * (v & 15);
        return ((atomicOr(&w[v >> 4], c << sh) >> sh) & 3u) == 0;
    }
};

// What a workgroup works on: its source's arrays.
template <bool LG, typename TT>
struct PlainCtx {
    const gint *rp, *col, *reach;
    int n;
    Codes<LG> lv;
    uint64_t *sg;   // path counts
    TT *tt;         // terms (FP64: the same words as sg, unless sg is kept)
    double *dl;     // dependencies of the source, when they are added in vertex order
    int32_t *S;     // vertices in level order
    int32_t *off;   // level offsets past LDS_LEVELS
    int32_t *drow;  // levels, when the source's row is kept
    PlainShared *sh;
    WaveRows *wr;   // this wave's
    WaveTerms *wt;  // (FP64 terms: its WaveSums)
    __device__ __forceinline__ int level_off(int l) const { return l < LDS_LEVELS ? sh->off[l] : off[l]; }
    __device__ __forceinline__ void set_off(int l, int x) const {
        if (l < LDS_LEVELS) sh->off[l] = x;
        else off[l] = x;
    }
};

// Row of flat arc g: the last k with P[k] <= g.
__device__ __forceinline__ int row_of(const WaveRows &r, int g) {
    int k = 0;
#pragma unroll
    for (int h = 32; h > 0; h >>= 1)
        if (r.P[k + h] <= g) k += h;
    return k;
}

// Lays the wave's rows (d arcs from j0 on each lane) out as one flat range;
// returns its length.
__device__ __forceinline__ int flat_rows(WaveRows &r, int j0, int d) {
    const int lane = threadIdx.x & 63;
    int inc = d;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(inc, o, 64);
        if (lane >= o) inc += y;
    }
    r.P[lane] = inc - d;
    r.A[lane] = j0 - (inc - d);
    r.acc[lane] = 0;
    psync();
    return __builtin_amdgcn_readlane(inc, 63);
}

// Appends the vertices that the wave's lanes took to level l+1's list.
template <int U, typename Ctx>
__device__ __forceinline__ void append(const Ctx &x, const int (&w)[U], const bool (&mine)[U], int q1,
                                       int *cnt) {
    uint64_t b[U];
    int tot = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        b[u] = pbal(mine[u]);
        tot += __popcll(b[u]);
    }
    if (tot == 0) return;
    int pos = 0;
    if ((threadIdx.x & 63) == 0) pos = atomicAdd(cnt, tot);
    pos = q1 + __builtin_amdgcn_readlane(pos, 0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if (mine[u]) x.S[prank(b[u], pos)] = w[u];
        pos += __popcll(b[u]);
    }
}

constexpr int PU = 4;  // arcs of a lane in flight
static_assert(sizeof(WaveTerms::t) >= 4 * 64 * PU, "a step's terms");

// Forward BFS from s.  Returns the deepest level, -1 when a uint64 count
// overflowed.
template <bool F64, typename Ctx>
__device__ __forceinline__ int plain_forward(const Ctx &x, int s, uint64_t limit) {
    const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63, wv = tid >> 6;
    PlainShared *sh = x.sh;
    for (int k = tid; k < (x.n + 15) / 16; k += nt) x.lv.w[k] = 0;
    if (x.drow)  // (a kept row tells the vertices that the source does not reach)
        for (int k = tid; k < x.n; k += nt) {
            x.drow[k] = BCX_INF;
            x.sg[k] = 0;
        }
    if (tid < 3) sh->cnt[tid] = sh->ovf[tid] = 0;
    pbarrier();
    if (tid == 0) {
        x.lv.take(s, 1);
        x.sg[s] = sig_one(F64);
        x.S[0] = s;
        x.set_off(0, 0);
        x.set_off(1, 1);
    }
    pbarrier();
    int q0 = 0, q1 = 1, l = 0;
    uint32_t cprev = 3, cnext = 2;  // codes of levels l-1 (l = 0: none set) and l+1
    while (true) {
        int *cnt = &sh->cnt[l % 3];
        // (last read two levels ago)
        if (tid == 0) sh->cnt[(l + 1) % 3] = sh->ovf[(l + 1) % 3] = 0;
        for (int base = q0 + wv * 64; base < q1; base += nt) {
            const int e = base + lane;
            int v = 0, j0 = 0, j1 = 0;
            if (e < q1) {
                v = x.S[e];
                j0 = x.rp[v];
                j1 = x.rp[v + 1];
            }
            const int d = j1 - j0;
            const uint64_t hubs = pbal(d > HUB);
            const int je = d > HUB ? j0 : j1;
            uint64_t acc = 0;
            double facc = 0.0;
            bool ovf = false;
            if (F64 || !pbal(d > SHORT)) {
                for (int j = j0; pbal(j < je); j += PU) {
                    int w[PU];
                    uint32_t f[PU];
                    uint64_t y[PU];
                    bool mine[PU];
#pragma unroll
                    for (int u = 0; u < PU; ++u) w[u] = j + u < je ? x.col[j + u] : -1;
#pragma unroll
                    for (int u = 0; u < PU; ++u) f[u] = x.lv.get(max(w[u], 0));
#pragma unroll
                    for (int u = 0; u < PU; ++u) y[u] = w[u] >= 0 && f[u] == cprev ? x.sg[w[u]] : 0;
#pragma unroll
                    for (int u = 0; u < PU; ++u) mine[u] = w[u] >= 0 && f[u] == 0 && x.lv.take(w[u], cnext);
#pragma unroll
                    for (int u = 0; u < PU; ++u) {
                        if (F64) facc += u2d(y[u]);
                        else ovf |= __builtin_add_overflow(acc, y[u], &acc);
                    }
                    append<PU>(x, w, mine, q1, cnt);
                }
            } else {
                WaveRows &r = *x.wr;
                const int T = flat_rows(r, j0, je - j0);
                for (int g0 = 0; g0 < T; g0 += 64 * PU) {
                    int w[PU], k[PU];
                    uint32_t f[PU];
                    uint64_t y[PU];
                    bool mine[PU];
#pragma unroll
                    for (int u = 0; u < PU; ++u) {
                        const int g = g0 + 64 * u + lane;
                        k[u] = row_of(r, g);
                        w[u] = g < T ? x.col[r.A[k[u]] + g] : -1;
                    }
#pragma unroll
                    for (int u = 0; u < PU; ++u) f[u] = x.lv.get(max(w[u], 0));
#pragma unroll
                    for (int u = 0; u < PU; ++u) y[u] = w[u] >= 0 && f[u] == cprev ? x.sg[w[u]] : 0;
#pragma unroll
                    for (int u = 0; u < PU; ++u) mine[u] = w[u] >= 0 && f[u] == 0 && x.lv.take(w[u], cnext);
                    append<PU>(x, w, mine, q1, cnt);
#pragma unroll
                    for (int u = 0; u < PU; ++u)
                        if (y[u]) {
                            const uint64_t old = atomicAdd((unsigned long long *)&r.acc[k[u]], (unsigned long long)y[u]);
                            ovf |= old + y[u] < old;
                        }
                }
                psync();
                acc = r.acc[lane];
                psync();
            }
            for (uint64_t m = hubs; m; m &= m - 1) {
                const int src = __ffsll((long long)m) - 1;
                const int a0 = __builtin_amdgcn_readlane(j0, src), a1 = __builtin_amdgcn_readlane(j1, src);
                uint64_t part = 0;
                double fsum = 0.0;
                for (int c = a0; c < a1; c += 64 * PU) {
                    int w[PU];
                    uint32_t f[PU];
                    uint64_t y[PU];
                    bool mine[PU];
#pragma unroll
                    for (int u = 0; u < PU; ++u) w[u] = c + 64 * u + lane < a1 ? x.col[c + 64 * u + lane] : -1;
#pragma unroll
                    for (int u = 0; u < PU; ++u) f[u] = x.lv.get(max(w[u], 0));
#pragma unroll
                    for (int u = 0; u < PU; ++u) y[u] = w[u] >= 0 && f[u] == cprev ? x.sg[w[u]] : 0;
#pragma unroll
                    for (int u = 0; u < PU; ++u) mine[u] = w[u] >= 0 && f[u] == 0 && x.lv.take(w[u], cnext);
                    append<PU>(x, w, mine, q1, cnt);
#pragma unroll
                    for (int u = 0; u < PU; ++u) {
                        if (F64) {  // in CSR order
                            for (uint64_t b = pbal(y[u] != 0); b; b &= b - 1)
                                fsum += u2d(prl64(y[u], __ffsll((long long)b) - 1));
                        } else {
                            ovf |= __builtin_add_overflow(part, y[u], &part);
                        }
                    }
                }
                if (!F64) {
#pragma unroll
                    for (int o = 32; o > 0; o >>= 1)
                        ovf |= __builtin_add_overflow(part, (uint64_t)__shfl_xor((unsigned long long)part, o, 64), &part);
                }
                if (lane == src) {
                    acc = part;
                    facc = fsum;
                }
            }
            if (e < q1) {
                if (l > 0) x.sg[v] = F64 ? d2u(facc) : acc;
                if (x.drow) x.drow[v] = l;
            }
            if (!F64 && pbal(ovf || (limit && acc >= limit && l > 0)) && lane == 0) sh->ovf[l % 3] = 1;
        }
        pbarrier();
        const int tail = q1 + *cnt;
        if (!F64 && sh->ovf[l % 3]) return -1;
        if (tail == q1) break;
        if (tid == 0) x.set_off(l + 2, tail);
        q0 = q1;
        q1 = tail;
        l++;
        const uint32_t c = cprev;  // l-1 <- l, l+1 <- l+2, whose code is the old l-1's
        cprev = 6 - cprev - cnext;
        cnext = c;
    }
    return l;
}

// Successor-method dependency, levels maxlvl .. 1; adds ws*delta to bc (and
// stores delta in probe, when given).  FP64 terms are summed in any order;
// compensated FP32 terms in CSR order, as every kernel of that precision does.
template <bool F64, bool LG, typename TT>
__device__ __forceinline__ void plain_backward(const PlainCtx<LG, TT> &x, int maxlvl, double ws, double *bc,
                                               double *probe) {
    constexpr bool ORD = sizeof(TT) == 4;
    using Acc = typename std::conditional<ORD, KahanP, SumP>::type;
    const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63, wv = tid >> 6;
    for (int l = maxlvl; l >= 1; --l) {
        const int q0 = x.level_off(l), q1 = x.level_off(l + 1);
        const uint32_t csucc = 1 + (uint32_t)((l + 1) % 3);
        for (int base = q0 + wv * 64; base < q1; base += nt) {
            const int e = base + lane;
            int v = 0, j0 = 0, j1 = 0, rv = 0;
            uint64_t sx = 0;
            if (e < q1) {
                v = x.S[e];
                j0 = x.rp[v];
                j1 = x.rp[v + 1];
                rv = x.reach[v];
                sx = x.sg[v];
            }
            Acc rho;
            if (l < maxlvl) {
                const int d = j1 - j0;
                const uint64_t hubs = pbal(d > HUB);
                const int je = d > HUB ? j0 : j1;
                if (!pbal(d > SHORT)) {
                    for (int j = j0; pbal(j < je); j += PU) {
                        int w[PU];
                        bool use[PU];
                        TT t[PU];
#pragma unroll
                        for (int u = 0; u < PU; ++u) w[u] = j + u < je ? x.col[j + u] : -1;
#pragma unroll
                        for (int u = 0; u < PU; ++u) use[u] = w[u] >= 0 && x.lv.get(max(w[u], 0)) == csucc;
#pragma unroll
                        for (int u = 0; u < PU; ++u) t[u] = use[u] ? x.tt[w[u]] : (TT)0;
#pragma unroll
                        for (int u = 0; u < PU; ++u)
                            if (use[u]) rho.add(t[u]);
                    }
                } else {
                    WaveRows &r = *x.wr;
                    const int T = flat_rows(r, j0, je - j0);
                    double *const sums = ((WaveSums *)x.wt)->s;
                    if constexpr (!ORD) {
#pragma unroll
                        for (int u = 0; u < 4; ++u) sums[64 * u + lane] = 0.0;
                        psync();
                    }
                    for (int g0 = 0; g0 < T; g0 += 64 * PU) {
                        int w[PU], k[PU];
                        bool use[PU];
                        TT t[PU];
#pragma unroll
                        for (int u = 0; u < PU; ++u) {
                            const int g = g0 + 64 * u + lane;
                            k[u] = row_of(r, g);
                            w[u] = g < T ? x.col[r.A[k[u]] + g] : -1;
                        }
#pragma unroll
                        for (int u = 0; u < PU; ++u) use[u] = w[u] >= 0 && x.lv.get(max(w[u], 0)) == csucc;
#pragma unroll
                        for (int u = 0; u < PU; ++u) t[u] = use[u] ? x.tt[w[u]] : (TT)0;
                        if constexpr (ORD) {
                            // the step's terms compacted in arc order, then
                            // each lane adds its row's
                            WaveTerms &q = *x.wt;
                            int tot = 0;
#pragma unroll
                            for (int u = 0; u < PU; ++u) {
                                const uint64_t b = pbal(use[u]);
                                const int at = prank(b, tot);
                                q.before[64 * u + lane] = (uint16_t)at;
                                if (use[u]) q.t[at] = t[u];
                                tot += __popcll(b);
                            }
                            if (lane == 0) q.before[64 * PU] = (uint16_t)tot;
                            psync();
                            const int p = r.P[lane], a0 = max(p - g0, 0), a1 = min(p + (je - j0) - g0, 64 * PU);
                            int i = 0, ie = 0;
                            if (a0 < a1) {
                                i = q.before[a0];
                                ie = q.before[a1];
                            }
                            for (; pbal(i < ie); i += 4) {
                                float y[4];
                                const int at = i < ie ? i : 0;
#pragma unroll
                                for (int u = 0; u < 4; ++u) y[u] = q.t[at + u];
#pragma unroll
                                for (int u = 0; u < 4; ++u) {
                                    Acc more = rho;
                                    more.add(y[u]);
                                    if (i + u < ie) rho = more;
                                }
                            }
                            psync();
                        } else {
#pragma unroll
                            for (int u = 0; u < PU; ++u)
                                if (use[u]) unsafeAtomicAdd(&sums[4 * k[u] + (lane & 3)], (double)t[u]);
                        }
                    }
                    if constexpr (!ORD) {
                        psync();
                        const double *s = &sums[4 * lane];
                        rho.s = (s[0] + s[1]) + (s[2] + s[3]);
                        psync();
                    }
                }
                for (uint64_t m = hubs; m; m &= m - 1) {
                    const int src = __ffsll((long long)m) - 1;
                    const int a0 = __builtin_amdgcn_readlane(j0, src), a1 = __builtin_amdgcn_readlane(j1, src);
                    Acc part;
                    for (int c = a0; c < a1; c += 64 * PU) {
                        int w[PU];
                        bool use[PU];
                        TT t[PU];
#pragma unroll
                        for (int u = 0; u < PU; ++u) w[u] = c + 64 * u + lane < a1 ? x.col[c + 64 * u + lane] : -1;
#pragma unroll
                        for (int u = 0; u < PU; ++u) use[u] = w[u] >= 0 && x.lv.get(max(w[u], 0)) == csucc;
#pragma unroll
                        for (int u = 0; u < PU; ++u) t[u] = use[u] ? x.tt[w[u]] : (TT)0;
#pragma unroll
                        for (int u = 0; u < PU; ++u) {
                            if constexpr (ORD) {
                                for (uint64_t b = pbal(use[u]); b; b &= b - 1)
                                    part.add(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(t[u]),
                                                                                      __ffsll((long long)b) - 1)));
                            } else {
                                part.add((double)t[u]);
                            }
                        }
                    }
                    if constexpr (!ORD) part.s = wave_sum(part.s);
                    if (lane == src) rho = part;
                }
            }
            if (e < q1) {
                const double sv = F64 ? u2d(sx) : (double)sx;
                const double sum = rho.value();
                const double delta = sv * sum;
                x.tt[v] = (TT)(((double)rv + 1.0) / sv + sum);
                if (x.dl) x.dl[v] = delta;
                else if (delta != 0.0) unsafeAtomicAdd(&bc[v], ws * delta);
                if (probe) probe[v] = delta;
            }
        }
        pbarrier();
    }
    if (!x.dl) return;
    // added in vertex order: neighbouring lanes' atomics share a line (a vertex
    // that the source does not reach has an earlier source's word)
    if (tid == 0) x.dl[x.S[0]] = 0.0;
    pbarrier();
    for (int v = tid; v < x.n; v += nt) {
        const double delta = x.lv.get(v) ? x.dl[v] : 0.0;
        if (delta != 0.0) unsafeAtomicAdd(&bc[v], ws * delta);
    }
}

// LDS of a workgroup past its static part: the waves' rows, then the codes
template <bool LG, typename TT>
__device__ __forceinline__ void carve(PlainCtx<LG, TT> &x, unsigned char *lds, const CompDev &c, uint32_t *lv_rows) {
    x.wr = (WaveRows *)(lds + (threadIdx.x >> 6) * wave_lds<TT>());
    x.wt = (WaveTerms *)(x.wr + 1);
    x.lv.w = LG ? lv_rows : (uint32_t *)(lds + (blockDim.x >> 6) * wave_lds<TT>());
    x.rp = glb(c.rp);
    x.col = glb(c.col);
    x.reach = glb(c.reach);
    x.n = c.n;
}

}  // namespace

template <bool F64, bool LG, typename TT>
__global__ __launch_bounds__(64 * PMAXW) void k_plain_bfs(CompDev c, PlainArgs a, PlainScratch sc, Rows rows) {
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ PlainShared sh;
    const int tid = threadIdx.x;
    const int64_t base = (int64_t)blockIdx.x * sc.stride;
    PlainCtx<LG, TT> x;
    // (a kept row holds its levels itself, so the workgroup's d row is free)
    carve<LG, TT>(x, lds, c, (uint32_t *)(sc.d + base));
    x.S = sc.S + base;
    x.off = sc.off + base;
    x.sh = &sh;
    double *bc = a.bc + (int64_t)(blockIdx.x % (unsigned)a.split) * c.n;
    while (true) {
        if (tid == 0) {
            sh.item = atomicAdd(&a.counters[0], 1);
            sh.stop = (!F64 && ald(&a.counters[1]) != 0) ? 1 : 0;
        }
        pbarrier();
        const int item = sh.item;
        if (sh.stop) return;  // (the component is redone)
        if (item >= a.count) break;
        const int s = a.src[item];
        const int slot = a.aux[item];
        const int mode = a.mode[item];
        const bool row = mode & MODE_ROW;
        x.sg = row ? rows.sig + (int64_t)slot * rows.stride : sc.sig + base;
        x.tt = row || sizeof(TT) == 4 ? (TT *)(sc.dl + base) : (TT *)x.sg;
        x.dl = row || !a.sweep ? nullptr : (sizeof(TT) == 4 ? (double *)x.sg : sc.dl + base);
        x.drow = row ? rows.d + (int64_t)slot * rows.stride : nullptr;
        const int maxlvl = plain_forward<F64>(x, s, a.limit);
        if (!F64 && maxlvl < 0) {
            if (tid == 0) atomicExch(&a.counters[1], 1);
            return;
        }
        if (tid == 0) atomicMax(&a.counters[2], maxlvl);
        if (mode & MODE_BC)
            plain_backward<F64>(x, maxlvl, (double)c.reach[s] + 1.0, bc, a.probe);
        pbarrier();
    }
}

template <bool F64, bool LG>
__global__ __launch_bounds__(64 * PMAXW) void k_plain_chain(CompDev c, ChainDev ch, PlainArgs a, PlainScratch sc,
                                                            Rows rows) {
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ PlainShared sh;
    __shared__ int hist[LDS_LEVELS + 2];
    const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63;
    const int64_t base = (int64_t)blockIdx.x * sc.stride;
    int32_t *d = sc.d + base, *off = sc.off + base;
    uint64_t *sg = sc.sig + base;
    PlainCtx<LG, double> x;
    carve<LG, double>(x, lds, c, (uint32_t *)(sc.dl + base));
    x.S = sc.S + base;
    x.off = off;
    x.sh = &sh;
    x.sg = sg;
    x.tt = a.probe ? a.probe + c.n : (double *)sg;
    x.dl = nullptr;
    x.drow = nullptr;
    while (true) {
        if (tid == 0) {
            sh.item = atomicAdd(&a.counters[0], 1);
            sh.top = 0;
        }
        pbarrier();
        const int item = sh.item;
        if (item >= a.count) break;
        const int ci = a.src[item], pos = a.aux[item];
        const int p0 = ch.ptr[ci], cnt = ch.ptr[ci + 1] - p0;
        const int s = ch.nodes[p0 + pos];
        const int ld = pos + 1, rd = cnt - pos;
        const int32_t *dL = rows.d + (int64_t)a.slots[2 * item] * rows.stride;
        const int32_t *dR = rows.d + (int64_t)a.slots[2 * item + 1] * rows.stride;
        const uint64_t *sL = rows.sig + (int64_t)a.slots[2 * item] * rows.stride;
        const uint64_t *sR = rows.sig + (int64_t)a.slots[2 * item + 1] * rows.stride;
        // combine (Codes/postprocesses.cu:329-351)
        int mymax = 0;
        for (int k = tid; k < c.n; k += nt) {
            const int a0 = dL[k], b0 = dR[k];
            const int la = a0 == BCX_INF ? BCX_INF : a0 + ld, lb = b0 == BCX_INF ? BCX_INF : b0 + rd;
            int lv;
            uint64_t sv;
            if (la < lb) { lv = la; sv = sL[k]; }
            else if (la > lb) { lv = lb; sv = sR[k]; }
            else { lv = lb; sv = F64 ? d2u(u2d(sL[k]) + u2d(sR[k])) : sL[k] + sR[k]; }
            d[k] = lv;
            sg[k] = sv;
            if (lv != BCX_INF) mymax = max(mymax, lv);
        }
        mymax = wave_max(mymax);
        if (lane == 0) atomicMax(&sh.top, mymax);
        for (int k = tid; k < (c.n + 15) / 16; k += nt) x.lv.w[k] = 0;
        pbarrier();
        // own chain: direct distances (Codes/postprocesses.cu:205-274, 354-360)
        for (int j = tid; j < cnt; j += nt) {
            const int y = ch.nodes[p0 + j];
            if (j == pos) {
                d[y] = 0;
                sg[y] = sig_one(F64);
                continue;
            }
            const int dist = j > pos ? j - pos : pos - j;
            if (d[y] > dist) {
                d[y] = dist;
                sg[y] = sig_one(F64);
            } else if (d[y] == dist) {
                sg[y] = F64 ? d2u(u2d(sg[y]) + 1.0) : sg[y] + 1;
            }
        }
        // final levels are BFS distances (< n); the combine maximum can be
        // larger on the source's own chain before the walk above fixes it
        const int maxl = min(sh.top, c.n - 1);
        // (a vertex that the endpoints do not reach lies past it and joins no level)
        const bool in_lds = maxl + 2 <= LDS_LEVELS;
        int *h = in_lds ? hist : off;  // off doubles as the histogram when deep
        for (int l = tid; l < maxl + 2; l += nt) h[l] = 0;
        pbarrier();
        // level codes and histogram; the lanes of a wave that share a level add
        // once (most of a small-world component sits on a few levels)
        for (int k0 = 0; k0 < c.n; k0 += nt) {
            const int k = k0 + tid;
            const int dk = k < c.n ? d[k] : -1, l = dk <= maxl ? dk : -1;
            if (l >= 0) x.lv.take(k, 1 + (uint32_t)(l % 3));
            for (uint64_t m = pbal(l >= 0); m;) {
                const int src = __ffsll((long long)m) - 1;
                const int l0 = __builtin_amdgcn_readlane(l, src);
                const uint64_t same = pbal(l == l0);
                if (lane == src) atomicAdd(&h[l0 + 1], __popcll(same));
                m &= ~same;
            }
        }
        pbarrier();
        if (tid == 0) {
            int run = 0;
            for (int l = 0; l < maxl + 2; ++l) {
                run += in_lds ? h[l] : ald(&h[l]);
                // start of level l (exclusive prefix over l+1 bins); the
                // cursors of a deep source overwrite off, which the sorted
                // list then gives back
                if (in_lds) {
                    h[l] = run;
                    x.set_off(l, run);
                } else {
                    ast(&h[l], run);
                }
            }
            sh.stop = run;  // vertices in the list
        }
        pbarrier();
        // h[l] now = number of vertices with level < l; use as cursors
        for (int k0 = 0; k0 < c.n; k0 += nt) {
            const int k = k0 + tid;
            const int dk = k < c.n ? d[k] : -1, l = dk <= maxl ? dk : -1;
            for (uint64_t m = pbal(l >= 0); m;) {
                const int src = __ffsll((long long)m) - 1;
                const int l0 = __builtin_amdgcn_readlane(l, src);
                const uint64_t same = pbal(l == l0);
                int at = 0;
                if (lane == src) at = atomicAdd(&h[l0], __popcll(same));
                at = __builtin_amdgcn_readlane(at, src);
                if (l == l0) x.S[prank(same, at)] = k;
                m &= ~same;
            }
        }
        pbarrier();
        if (!in_lds) {
            // every level's offset again from the sorted levels (the first
            // LDS_LEVELS of them in LDS)
            const int total = sh.stop;
            if (tid == 0) x.set_off(0, 0);
            for (int i = tid; i < total; i += nt) {
                const int li = d[x.S[i]];
                const int lp = i ? d[x.S[i - 1]] : -1;
                for (int l = lp + 1; l <= li; ++l) x.set_off(l, i);
                if (i == total - 1)
                    for (int l = li + 1; l <= maxl + 1; ++l) x.set_off(l, total);
            }
            pbarrier();
        }
        // the deepest non-empty level
        int top = maxl;
        while (top > 0 && x.level_off(top) == x.level_off(top + 1)) --top;
        if (tid == 0) atomicMax(&a.counters[2], top);
        plain_backward<F64>(x, top, (double)c.reach[s] + 1.0, a.bc, a.probe);
        pbarrier();
    }
}

// Whether the sources' dependencies are stored and added to BC in vertex order,
// a line's atomics together, instead of one by one as the backward makes them.
// Sparse components have an atomic per few arcs (a grid of 26k: 330M for 16384
// sources, two thirds of the bytes written); the row of dependencies costs cache
// that larger components need.  One by one / in order: grids of 3.7k, 11k, 18.6k,
// 22k and 26k vertices 1431 / 1261, 2553 / 2283, 3516 / 3176, 3973 / 3939 and
// 25900 / 31000 us; power-law cores of 12.7k and 16.9k 1857 / 1894 and 2357 /
// 2538; R-MAT core of 12k 7890 / 8084.
bool plain_sweep(int32_t n, int64_t arcs) { return n <= 20000 && arcs <= 5 * (int64_t)n; }

// Waves per source by the component's size: a barrier per level against the
// vertices a level gives the waves.  4 / 8 / 16 waves (us; k sources): grid of
// 3.7k vertices, k 2049: 1370 / 1485 / 2654; grid of 18.6k, k 2049: 5150 / 5100 /
// 7540; power-law core of 21k, k 2000: 6837 / 5351 / 6150, of 84k, k 1000: 26150 /
// 21440 / 18950, of 335k, k 600: 82052 / 56163 / 46738; R-MAT core of 86k, k 1000:
// 31553 / 30536 / 25703; grid of 74k, k 2049: 15381 / 14186 / 14663.  One or two
// 16-wave workgroups per compute unit run the same.
PlainShape plain_shape(int32_t n, bool fp32) {
    PlainShape p;
    p.waves = n <= 8192 ? 4 : (n <= 49152 ? 8 : 16);
    p.lds_codes = n <= LV_LDS_N;
    const int64_t codes = p.lds_codes ? 4 * (((int64_t)n + 15) / 16) : 0;
    p.lds = (int)codes + p.waves * (fp32 ? wave_lds<float>() : wave_lds<double>());
    const int64_t fit = 160 * 1024 / (p.lds + (int64_t)sizeof(PlainShared) + 4 * (LDS_LEVELS + 2) + 512);
    p.per_cu = (int)std::max<int64_t>(1, std::min<int64_t>(fit, 24 / p.waves));
    return p;
}

hipError_t launch_plain_bfs(const CompDev &c, const PlainArgs &a, const PlainScratch &sc, const Rows &rows,
                            const PlainShape &p, int grid, hipStream_t st) {
    const dim3 g(grid), b(64 * p.waves);
    if (a.fp32 && !a.sigma_f64) {
        if (p.lds_codes) hipLaunchKernelGGL((k_plain_bfs<false, false, float>), g, b, p.lds, st, c, a, sc, rows);
        else hipLaunchKernelGGL((k_plain_bfs<false, true, float>), g, b, p.lds, st, c, a, sc, rows);
    } else if (a.sigma_f64) {
        if (p.lds_codes) hipLaunchKernelGGL((k_plain_bfs<true, false, double>), g, b, p.lds, st, c, a, sc, rows);
        else hipLaunchKernelGGL((k_plain_bfs<true, true, double>), g, b, p.lds, st, c, a, sc, rows);
    } else {
        if (p.lds_codes) hipLaunchKernelGGL((k_plain_bfs<false, false, double>), g, b, p.lds, st, c, a, sc, rows);
        else hipLaunchKernelGGL((k_plain_bfs<false, true, double>), g, b, p.lds, st, c, a, sc, rows);
    }
    return hipGetLastError();
}

__global__ void k_plain_fold(double *bc, const double *copies, const int32_t *perm, int n, int split) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= n) return;
    ExactSum s;
    for (int k0 = 0; k0 < split; k0 += 8) {  // (eight loads in flight)
        double x[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) x[k] = k0 + k < split ? copies[(int64_t)(k0 + k) * n + v] : 0.0;
#pragma unroll
        for (int k = 0; k < 8; ++k) s.add(x[k]);
    }
    bc[perm ? perm[v] : v] += s.value();
}

hipError_t launch_plain_fold(double *bc, const double *copies, const int32_t *perm, int n, int split, hipStream_t st) {
    hipLaunchKernelGGL(k_plain_fold, dim3((n + 255) / 256), dim3(256), 0, st, bc, copies, perm, n, split);
    return hipGetLastError();
}

// One wave per row.
__global__ __launch_bounds__(256) void k_plain_reorder(CompDev from, CompDev to, const int32_t *perm,
                                                       const int32_t *inv) {
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (i >= from.n) return;
    const int v = perm[i], a = from.rp[v], d = from.rp[v + 1] - a, at = to.rp[i];
    for (int j = lane; j < d; j += 64) const_cast<int32_t *>(to.col)[at + j] = inv[from.col[a + j]];
    if (lane == 0) const_cast<int32_t *>(to.reach)[i] = from.reach[v];
}

hipError_t launch_plain_reorder(const CompDev &from, const CompDev &to, const int32_t *perm, const int32_t *inv,
                                hipStream_t st) {
    hipLaunchKernelGGL(k_plain_reorder, dim3((from.n + 3) / 4), dim3(256), 0, st, from, to, perm, inv);
    return hipGetLastError();
}

hipError_t launch_plain_chain(const CompDev &c, const ChainDev &ch, const PlainArgs &a, const PlainScratch &sc,
                              const Rows &rows, const PlainShape &p, int grid, hipStream_t st) {
    const dim3 g(grid), b(64 * p.waves);
    if (p.lds_codes && a.sigma_f64)
        hipLaunchKernelGGL((k_plain_chain<true, false>), g, b, p.lds, st, c, ch, a, sc, rows);
    else if (p.lds_codes) hipLaunchKernelGGL((k_plain_chain<false, false>), g, b, p.lds, st, c, ch, a, sc, rows);
    else if (a.sigma_f64) hipLaunchKernelGGL((k_plain_chain<true, true>), g, b, p.lds, st, c, ch, a, sc, rows);
    else hipLaunchKernelGGL((k_plain_chain<false, true>), g, b, p.lds, st, c, ch, a, sc, rows);
    return hipGetLastError();
}

}  // namespace bcx
