// Internal launch interface of the FP64 MFMA GEMM (gemm_f64.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.hpp"

namespace dtcf {

// Operand addressing modes (rows of the view x k):
//   kDK : dense, (r, c) at r*ld + c   -- k contiguous
//   kDMN: dense, (r, c) at c*ld + r   -- rows contiguous
//   kVK : offset tables, pairs (c, c+1) contiguous
//   kVMN: offset tables, pairs (r, r+1) contiguous
enum { kDK = 0, kDMN = 1, kVK = 2, kVMN = 3 };

// Tile configurations (BM x BN), selectable per launch by the autotuner.
// 192x64 and 64x192 serve thin results (one side at most 64) with long K:
// a 64-wide tile of the thin side, three times as deep on the other, so
// the thin operand is re-read by a third as many tiles as with 64 x 64.
// kCfgThin is the streaming kernel for thin results (one side at most 48,
// or 192 with K <= 48) with short K (thin_f64_launch); shapes it does not
// take run 64 x 64 tiles.  The grouped launch takes the first four.
enum {
    kCfg128x128 = 0,
    kCfg192x96 = 1,
    kCfg96x192 = 2,
    kCfg64x64 = 3,
    kCfg192x64 = 4,
    kCfg64x192 = 5,
    kCfgThin = 6,
    kCfgCount = 7,
    kCfgGroupCount = 4
};
// The C tile configuration dtcf_gemm_* uses for an m x n x k GEMM.
int pick_config(int64_t m, int64_t n, int64_t k, bool gather = false);

struct OpArgs {
    int64_t ld;
    const int64_t *rofs;
    const int64_t *cofs;
    const int64_t *blk;
    FastDiv div_rpb, div_cpb;
    int64_t ncb;
    int32_t vec2;  // 1: (r,c),(r,c+1) [k-mode] or (r,c),(r+1,c) [mn-mode] are adjacent
                   //    and 16-byte aligned wherever both are in range (c or r even)
    int32_t adj;   // views: 1: they are adjacent, at any alignment
    int32_t gather;  // views: 1: single elements whose neighbours lie elsewhere
};

struct GemmArgs {
    int64_t m, n, k;
    double alpha;
    const double *A;
    const double *B;
    double *C;
    OpArgs a, b, c;
    int32_t amode, bmode, cview;
    uint32_t tiles_m, tiles_n;
    int64_t nfast;  // K steps loaded without bounds checks (gemm_tile.hpp)
    // Split tiles: workgroups [0, t_full) own whole tiles; the K steps of the
    // tiles from t_full on, `steps` in all, are cut into `sw` equal runs, one
    // per workgroup (SplitPlan).
    uint32_t t_full, sw;
    int64_t steps;
    double *ws;
    // 0: C += alpha * A * B (every reference call site); 1: C = alpha * A * B
    // (C is neither cleared first nor read)
    int32_t overwrite;
};

int gemm_f64_launch(GemmArgs g, int cfg, hipStream_t s);

// Up to kGroupMax independent dense GEMMs C_p (+)= alpha * op(A_p) * op(B_p)
// in one launch, every problem with the same operand layouts: A_p m x k
// (kDK) or k x m (kDMN), B_p n x k (kDK) or k x n (kDMN); C_p row-major.
// tiles_m, tiles_n, t_whole, nfast, wg0, tail0 and step0 are filled in by the
// launch: problem p's tiles [0, t_whole) run whole, in workgroups wg0[p]..,
// its tiles [t_whole, tiles) are the split tiles tail0[p].. of the launch,
// whose K steps are the steps step0[p].. of the `steps` that `sw` workgroups
// share (as in GemmArgs).  A problem without whole (split) tiles has the wg0
// (tail0, step0) of the next, and entries past the last problem hold the
// largest value, so the last entry not above a workgroup, tile or step is its
// problem: one load of neighbouring words and as many compares.
constexpr int kGroupMax = 16;
struct GemmGroupProb {
    int64_t m, n, k;
    const double *A;
    const double *B;
    double *C;
    int64_t lda, ldb, ldc;
    int32_t vec2a, vec2b;
    uint32_t tiles_m, tiles_n, t_whole;
    int64_t nfast;
};
struct GemmGroupArgs {
    double alpha;
    int32_t overwrite;
    int32_t np;
    uint32_t wg_whole, sw;  // workgroups of whole tiles; runs of split tiles
    int64_t steps;
    double *ws;
    uint32_t wg0[kGroupMax], tail0[kGroupMax];
    int64_t step0[kGroupMax];
    GemmGroupProb p[kGroupMax];
};

// One instantiation per C tile (gemm_tile_*.hip).
int gemm_tile_128x128(const GemmArgs &g, hipStream_t s);
int gemm_tile_192x96(const GemmArgs &g, hipStream_t s);
int gemm_tile_96x192(const GemmArgs &g, hipStream_t s);
int gemm_tile_64x64(const GemmArgs &g, hipStream_t s);
int gemm_tile_192x64(const GemmArgs &g, hipStream_t s);
int gemm_tile_64x192(const GemmArgs &g, hipStream_t s);
int gemm_group_tile_128x128(const GemmGroupArgs &ga, int amode, int bmode, hipStream_t s);
int gemm_group_tile_192x96(const GemmGroupArgs &ga, int amode, int bmode, hipStream_t s);
int gemm_group_tile_96x192(const GemmGroupArgs &ga, int amode, int bmode, hipStream_t s);
int gemm_group_tile_64x64(const GemmGroupArgs &ga, int amode, int bmode, hipStream_t s);
// How a launch of T tiles of nk K steps each fills the device: the last
// `nsplit` tiles are cut over K.  Their nsplit * nk steps, tile after tile,
// are dealt in `sw` equal runs to as many workgroups.  A run that covers a
// whole tile writes C; the piece of a tile at the start of run w goes to
// workspace slot 2 w, one at its end (when it is not also the start) to 2 w
// + 1, and a second kernel adds each tile's pieces to C in K order.  `us` is
// the predicted time, which also chooses between tiles (pick_config).
struct SplitPlan {
    uint32_t nsplit = 0, sw = 0;
    double us = 0.0;
};
// What the prediction knows of a C tile: us per K step of a workgroup when
// a CU's matrix cores are busy, workgroups per CU, and the share of the CU's
// rate that 1, 2, .. workgroups reach.  even: only cuts of every split tile
// into equal runs, which keep the workgroups on a few common K positions (a
// kernel whose operand panels must be shared through the L2s).
struct TileRate {
    int bm, bn, occ;
    double step_us, share[4];
    bool even = false;
    double cut_us = 4.0;  // what any cut costs beside its pieces
};
TileRate tile_rate(int cfg, bool gather = false);
// panel: rows of A and B together that one K step of the whole product
// reads (tiles_m bm + tiles_n bn, 0: much shared, as in a large product).
SplitPlan gemm_split_plan(uint32_t T, int64_t nk, int64_t panel, int cus, const TileRate &t);

int gemm_f64_group_launch(const GemmGroupArgs &ga, int cfg, int amode, int bmode, hipStream_t s);

// Matrix-vector products inside the view GEMM: y(r) (+)= alpha * sum_c
// M(r, c) x(c) over the rows of a view M whose column pairs are adjacent and
// 16-byte aligned (no block table), x a 1 x k view, y the single column
// (ycol = 1: y(r) = Y(r, 0)) or single row (ycol = 0: y(r) = Y(0, r)) of a
// dense Y (pitch ldy) or of a view.  k <= kGemvMaxK (x is staged in LDS).
constexpr int64_t kGemvMaxK = 20480;
struct GemvArgs {
    int64_t rows, k;
    double alpha;
    const double *M;
    const int64_t *mrofs, *mcofs;
    const double *X;
    OpArgs xv;
    double *Y;
    OpArgs yv;
    int32_t yview, ycol, overwrite;
    int64_t ldy;
};
int gemv_f64_launch(const GemvArgs &g, hipStream_t s);
// The same product when M has its row pairs adjacent instead (rofs[r + 1] =
// rofs[r] + 1 for even r, offsets even, rows even, M 16-byte aligned): any k.
int gemv_rows_f64_launch(const GemvArgs &g, hipStream_t s);

// Thin products: one side of C at most kThinMaxWidth wide (or at most
// kThinMaxWide with K <= kThinWideK), the other long (rows), K a multiple
// of 8 and short enough that the thin operand's K x width fragments and the
// offsets fit kThinLdsBytes of LDS.  thin_shape is the shape test; the
// launch also needs the long operand's pairs adjacent and 16-byte aligned
// (vec2), no block table on it or on a C view, and returns kThinDecline
// otherwise.
constexpr int64_t kThinMaxWidth = 48;
constexpr int64_t kThinMaxWide = 192;
constexpr int64_t kThinWideK = 48;
constexpr int64_t kThinLdsBytes = 80 * 1024;
constexpr int kThinDecline = 1;
bool thin_shape(int64_t m, int64_t n, int64_t k, int64_t min_rows);
int thin_f64_launch(const GemmArgs &g, hipStream_t s);

// Allocates the split workspace of stream `s` at the largest size any
// GEMM on it can need, so later launches on `s` never allocate.
int gemm_reserve_workspace(hipStream_t s);
// The split workspace of stream `s` (grown to `need` bytes if smaller; work
// on one stream shares it in stream order), and the device's CU count.
// A capturing stream cannot grow its own: with at least `uncut` bytes *ws is
// null and the launch runs without cuts, with less the call is refused.
int gemm_workspace(hipStream_t s, size_t need, double **ws, size_t uncut = SIZE_MAX);
// The `uncut` of T tiles (tile elements each) of nk K steps on `slots`
// resident workgroups: 0 where whole tiles fill most of every round, else what
// filling them by even cuts takes, since uncut such a product leaves up to
// nearly all of the device idle.
size_t gemm_uncut_bytes(uint32_t T, uint32_t slots, int64_t nk, size_t tile);
int gemm_device_cus(int *cus);

// dtcf_gemm_view_f64 with C = alpha * A * B instead of C += (capi.hip).
int gemm_view_overwrite(int64_t m, int64_t n, int64_t k, double alpha, const double *A,
                        dtcf_view av, const double *B, dtcf_view bv, double *C, dtcf_view cv,
                        int64_t ldc, hipStream_t stream);

// Slice products (mixed.hip): dtcf_gemm_split_f64 with C = alpha * A * B^T
// instead of C += when overwrite is set, which needs a fused kernel for
// (prec, nslice, level): gemm_split_fused.
bool gemm_split_fused(int prec, int ns, int lev);
int gemm_split_f64_impl(int prec, int nslice, int64_t m, int64_t n, int64_t k, double alpha,
                        const void *A_slices, const int32_t *ea, const void *B_slices,
                        const int32_t *eb, int max_level, double *C, dtcf_view cv, int64_t ldc,
                        void *stream, int overwrite);

}  // namespace dtcf
