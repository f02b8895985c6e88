// Wave-per-source kernel for small components: device view and launcher.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bcx_small.h"

namespace bcx {

// LDS of a workgroup.  Shared by its waves: the component's BC accumulator
// (8 B per vertex), row pointers (4 B) and columns (2 B per arc), rows padded to
// groups of four arcs with one empty group at the end.
// Per wave, i.e. per source in flight: one 8-byte word per vertex (the path
// count, which the backward overwrites with the vertex's term), a level code
// (1 B) and the level-ordered vertex list (2 B), each with two more entries
// that lanes without an arc of their own read and write.
constexpr int SRC_N = 2048;                 // largest component (list entries are 15-bit ids and a flag)
constexpr int SRC_WAVES = 16;               // waves of a workgroup
constexpr int64_t SRC_LDS = 160 * 1024 - 512;  // dynamic LDS of a workgroup at most
constexpr int SRC_COPIES = 16;              // BC accumulators of a launch with FP64 terms

__host__ __device__ constexpr int64_t src_up16(int64_t x) { return (x + 15) & ~(int64_t)15; }
// (groups: sum over the rows of ceil(arcs / 4))
__host__ __device__ constexpr int64_t src_shared_bytes(int64_t n, int64_t groups) {
    return src_up16(8 * n) + src_up16(4 * (n + 1)) + src_up16(8 * (groups + 1));
}
__host__ __device__ constexpr int64_t src_wave_bytes(int64_t n) {
    return src_up16(8 * (n + 2)) + src_up16(n + 2) + src_up16(2 * (n + 2));
}
// Sources in flight in a workgroup of `lds` dynamic bytes.
__host__ __device__ constexpr int64_t src_waves(int64_t n, int64_t groups, int64_t lds) {
    const int64_t w = (lds - src_shared_bytes(n, groups)) / src_wave_bytes(n);
    return w < 0 ? 0 : (w > SRC_WAVES ? SRC_WAVES : w);
}

// BC accumulators of a workgroup with FP64 terms: 4, 2 or 1, those past the first
// in what its waves leave of `lds`.  A wave adds to one of them, so a tile may be
// that much wider for the same rounding (400 components of 3 to 2000 vertices and a
// core, whole run: 7.40 ms with one, 7.25 so; a fifth of it: 1198 and 1150 us).
__host__ __device__ constexpr int src_accs(int64_t n, int64_t groups, int64_t lds) {
    const int64_t rest = lds - src_shared_bytes(n, groups) - src_waves(n, groups, lds) * src_wave_bytes(n);
    return rest >= 3 * src_up16(8 * n) ? 4 : (rest >= src_up16(8 * n) ? 2 : 1);
}

struct SrcArgs {
    const SmallComp *comps;
    const SmallTile *tiles;  // at most 64 sources each
    int32_t n_tiles;
    int32_t lds;             // dynamic LDS bytes of the launch
    const int32_t *srcs;
    const double *ws;
    int32_t *counter;        // [0] work counter, [1] tiles listed for an FP64 rerun, [2] deepest level
    int32_t *redo;           // [n_tiles] those tiles
    uint64_t limit;          // u64 path-count threshold (0 = 2^64)
    int32_t stop;            // take no further tile once one has overflowed
    // FP64 terms: words from one of SRC_COPIES accumulators to the next (0:
    // there is one); launch_src_fold adds them up
    int64_t copy;
    // probe only (null in runs): [n][64] per (vertex, source) of the last tile
    uint64_t *psig;
    int32_t *lvl;
    double *dbg;
    const int32_t *n_tiles_dev;  // when set, read instead of n_tiles
};

hipError_t launch_src(const SrcArgs &a, bool f64, bool fp32, int grid, hipStream_t st);
// The sum of the accumulators into the first, over n words from bc, and into out
// (optional, host memory); clears the others.  ctr (optional): three counters that
// go to ctr_out.
hipError_t launch_src_fold(double *bc, int64_t copy, int64_t n, double *out, const int32_t *ctr, int32_t *ctr_out,
                           hipStream_t st);
int src_blocks_per_cu(int lds);

}  // namespace bcx
