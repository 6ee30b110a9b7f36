// K-step runs of the split tiles of a GEMM launch (SplitPlan in
// gemm_f64.hpp): which steps a run holds, and the sum of a tile's pieces.
#pragma once
#include "common.hpp"

namespace dtcf {
namespace {

// First K step of run w of `sw` over `steps` (sw <= steps: no run is empty),
// and the run that holds step s.
// A 64-bit division is about a microsecond of a workgroup's start: 32 bits
// where they hold.
__device__ inline int64_t div_small(int64_t a, int64_t b)
{
    return ((a | b) >> 32) == 0 ? (int64_t)((uint32_t)a / (uint32_t)b) : a / b;
}
__device__ inline int64_t run_begin(uint32_t w, uint32_t sw, int64_t steps) { return div_small(w * steps, sw); }
__device__ inline uint32_t run_of(int64_t s, uint32_t sw, int64_t steps)
{
    return (uint32_t)div_small((s + 1) * sw - 1, steps);
}

// Run index of a workgroup past the whole tiles: neighbouring runs, which
// share tiles and operand panels, go to one XCD.
__device__ inline uint32_t run_index(uint32_t i, uint32_t sw) { return (sw & 7u) ? i : (i & 7u) * (sw >> 3) + (i >> 3); }

// The pieces of a tile whose K steps are [s0, s0 + nk) of the split ones,
// element e, added in K order (whole: one run covers the tile and wrote C).
// One element per thread: the reduce is bound by the latency of its loads,
// and four elements per thread (a quarter of the workgroups) took 15.7
// instead of 13.3 us with the product at 1024 x 64 x 1024.
__device__ inline double sum_runs(const double *ws, int64_t s0, int64_t nk, uint32_t sw, int64_t steps,
                                  int64_t tile, int e, bool &whole)
{
    const uint32_t w0 = run_of(s0, sw, steps), w1 = run_of(s0 + nk - 1, sw, steps);
    whole = w0 == w1;
    if (whole) return 0.0;
    const double first = ws[(2 * (int64_t)w0 + (run_begin(w0, sw, steps) < s0)) * tile + e];
    return sum_in_order(ws + 2 * ((int64_t)w0 + 1) * tile + e, w1 - w0, 2 * tile, first);
}

// The pieces of tile t of `tiles` split ones of nk K steps each, element e,
// added in K order (whole: one run covers the tile and wrote C).  Where the
// runs are even cuts of every tile, its slots follow from one division instead
// of the runs' ends (120 tiles of 128 x 128 in two: 14.2 -> 12.5 us).
__device__ inline double sum_pieces(const double *ws, uint32_t t, uint32_t tiles, int64_t nk, uint32_t sw,
                                    int64_t steps, int64_t tile, int e, bool &whole)
{
    const uint32_t per = sw / tiles;
    if (per * tiles != sw) return sum_runs(ws, t * nk, nk, sw, steps, tile, e, whole);
    whole = per == 1;
    if (whole) return 0.0;
    const double *w = ws + 2 * (int64_t)(t * per) * tile + e;
    return sum_in_order(w + 2 * tile, per - 1, 2 * tile, *w);
}

}  // namespace
}  // namespace dtcf
