// FP64 GEMM on the gfx950 matrix cores (v_mfma_f64_16x16x4_f64): tile
// choice by configuration, the K-split rule and the split workspaces.
//
// Replaces the dgemm behind local_contraction (localcontract.cc:3-21) and
// DLTC compute (DLTC/compute.cc:3-36).  One kernel template (gemm_tile.hpp)
// serves the plain row-major GEMM and the fused form where operands are
// read straight out of the permuted tile storage through dtcf_view offset
// tables (the create_big_matrix pack of transpose_helper.cc:20-171 is never
// materialised).
//
// MFMA operand layout (16x16x4 f64, wave64): lane l holds A[l%16][l/16] and
// B[l/16][l%16]; the result holds D[l/16 + 4*r][l%16] in element r (checked
// on the device by tests/test_gpu_core.py::test_mfma_layout_single_block).
//
// Workgroup ids are remapped so consecutive C tiles of a row group land on
// the same XCD (its own L2), then swizzled in groups of 8 tile rows.
//
// Shapes the tiles serve badly have streaming kernels of their own, chosen
// by the launch (gemm_stream.hip).
#include <algorithm>
#include <map>
#include <mutex>

#include "common.hpp"
#include "gemm_f64.hpp"

namespace dtcf {
namespace {

// CU count per device, and the split workspace per (device, stream):
// GEMMs enqueued on different streams never share a workspace; GEMMs on one
// stream are ordered by it.
std::mutex g_dev_mu;
int g_cus[64];
std::map<std::pair<int, hipStream_t>, std::pair<double *, size_t>> g_ws;

int device_cus(int *cus)
{
    int d = 0;
    DTCF_HIP(hipGetDevice(&d));
    DTCF_REQUIRE(d >= 0 && d < 64, "gemm: device index out of range");
    std::lock_guard<std::mutex> lk(g_dev_mu);
    if (g_cus[d] == 0) {
        int c = 0;
        DTCF_HIP(hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, d));
        g_cus[d] = c > 0 ? c : 1;
    }
    *cus = g_cus[d];
    return DTCF_OK;
}

int split_workspace(hipStream_t s, size_t need, size_t uncut, double **ws)
{
    int d = 0;
    DTCF_HIP(hipGetDevice(&d));
    std::lock_guard<std::mutex> lk(g_dev_mu);
    auto &e = g_ws[std::make_pair(d, s)];
    if (e.second < need) {
        // growing allocates (and frees the old buffer): never inside a graph
        // capture, where the allocation would run outside the graph and the
        // free could release a buffer an earlier graph still uses
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        DTCF_HIP(hipStreamIsCapturing(s, &cs));
        if (cs != hipStreamCaptureStatusNone) {
            if (e.second >= uncut) {
                *ws = nullptr;
                return DTCF_OK;
            }
            set_error("gemm: the split-K workspace of a capturing stream must be reserved before "
                      "capture (dtcf_gemm_reserve_workspace)");
            return DTCF_ERR_INVALID;
        }
        if (e.first) DTCF_HIP(hipStreamSynchronize(s));  // the old buffer may be in use
        if (e.first) (void)hipFree(e.first);
        e.first = nullptr;
        e.second = 0;
        DTCF_HIP(hipMalloc(&e.first, need));
        e.second = need;
    }
    *ws = e.first;
    return DTCF_OK;
}

}  // namespace

TileRate tile_rate(int cfg, bool gather)
{
    // Measured with whole tiles, one to four workgroups on every CU: 256,
    // 512 and 1024 tiles of 64 x 64 x 4096 in 195, 278 and 515 us, 256 and
    // 512 tiles of 128 x 128 in 561 (x 4096) and 514 us (x 2048).
    TileRate t;
    switch (cfg) {
    case kCfg192x96: t = {192, 96, 2, 2.25, {0.88, 1.0, 1.0, 1.0}}; break;
    case kCfg96x192: t = {96, 192, 2, 2.25, {0.88, 1.0, 1.0, 1.0}}; break;
    case kCfg64x64: t = {64, 64, 4, 0.50, {0.66, 0.925, 0.98, 1.0}}; break;
    case kCfg192x64: t = {192, 64, 2, 1.52, {0.85, 1.0, 1.0, 1.0}}; break;
    case kCfg64x192: t = {64, 192, 2, 1.52, {0.85, 1.0, 1.0, 1.0}}; break;
    default: t = {128, 128, 2, 1.96, {0.895, 1.0, 1.0, 1.0}}; break;
    }
    // An operand read element by element from lines of its own: the CU's loads
    // bound the step, 1.4 us on 64 x 64 tiles from two workgroups on and 4.5 on
    // 128 x 128, and lines serve several steps and tiles only from the L2s, so
    // the cuts are even (SplitPlan).  us, rated as pairs / so: 152 x 1295 x
    // 756 41.3 / 27.5, 782 x 700 x 450 49.4 / 33.1, 176 x 630 x 910 29.5 / 21.8.
    if (gather) {
        t.step_us *= t.bm * t.bn <= 64 * 64 ? 2.8 : 2.3;
        t.share[0] = t.bm * t.bn <= 64 * 64 ? 0.7 : 1.0;
        for (int c = 1; c < 4; c++) t.share[c] = 1.0;
        t.even = true;
    }
    return t;
}

SplitPlan gemm_split_plan(uint32_t T, int64_t nk, int64_t panel, int cus, const TileRate &t)
{
    const uint32_t slots = (uint32_t)cus * t.occ;
    const double step = t.step_us;
    // c workgroups on the busiest CU, each running `n` steps.  A step that
    // reads `hbm` bytes no other tile reads (thin results with long K) is
    // bound by HBM instead, or, with too few workgroups to hide it, by its
    // latency: 32 x 32 x 524288 took 148 us in 256 runs and 104 in 512, 128 x
    // 128 x 131072 105 and 92.
    const double hbm = (double)panel * 16 * 8 / T, all = (double)(t.bm + t.bn) * 16 * 8;
    auto run_us = [&](double n, uint32_t c) {
        const double mfma = step * c / t.share[std::min<uint32_t>(c, 4) - 1];
        const double lat = 2.5 * std::min(1.0, hbm / all);
        return n * std::max({mfma, hbm * c * cus / 5.0e6, lat});
    };
    SplitPlan best;
    const double whole = (double)(T / slots) * t.occ * nk * step;
    const uint32_t R = T % slots;
    best.us = whole;
    if (R == 0) return best;
    best.us += run_us((double)nk, (R + cus - 1) / cus);
    const int64_t steps = (int64_t)R * nk;
    // Starting workgroups takes about 12 ns each (1 / 8 of an XCD's 0.1 us).
    // Splitting pays a second launch (4 us), writes and reads back its pieces
    // (16 B per element at about 6 TB/s, L2 and the MALL helping) and waits
    // for eight of a tile's pieces at a time.
    best.us += 0.012 * R;
    auto consider = [&](uint32_t W, double pieces) {
        const double n = (double)((steps + W - 1) / W);
        const double us = whole + run_us(n, (W + cus - 1) / cus) + 0.012 * W + t.cut_us +
                          pieces * t.bm * t.bn * 16.0 / 6.0e6 + 0.7 * (pieces / R / 8.0 + 1.0);
        if (us < best.us) {
            best.us = us;
            best.nsplit = R;
            best.sw = W;
        }
    };
    // Runs of at least four steps: one, two, .. workgroups on every CU, and
    // the even cuts of each tile, which leave fewer pieces.
    for (int c = 1; c <= t.occ && !t.even; c++)
        if (steps >= 4 * (int64_t)cus * c) consider((uint32_t)cus * c, (double)R + (double)cus * c);
    for (uint32_t c = 2; c <= 512 && (uint64_t)R * c <= slots && nk >= 4 * (int64_t)c; c++)
        consider(R * c, (double)R * c);
    return best;
}

int gemm_f64_group_launch(const GemmGroupArgs &ga, int cfg, int amode, int bmode, hipStream_t s)
{
    DTCF_REQUIRE(ga.np >= 0 && ga.np <= kGroupMax, "gemm group: too many problems");
    for (int i = 0; i < ga.np; i++)
        DTCF_REQUIRE(ga.p[i].m > 0 && ga.p[i].n > 0 && ga.p[i].k > 0, "gemm group: empty problem");
    if (ga.np == 0) return DTCF_OK;
    switch (cfg) {
    case kCfg128x128: return gemm_group_tile_128x128(ga, amode, bmode, s);
    case kCfg192x96: return gemm_group_tile_192x96(ga, amode, bmode, s);
    case kCfg96x192: return gemm_group_tile_96x192(ga, amode, bmode, s);
    case kCfg64x64: return gemm_group_tile_64x64(ga, amode, bmode, s);
    default: break;
    }
    set_error("gemm group: unknown tile configuration");
    return DTCF_ERR_INVALID;
}

int gemm_workspace(hipStream_t s, size_t need, double **ws, size_t uncut) { return split_workspace(s, need, uncut, ws); }

// The last partial round of at most half the slots, or a grid under half of
// them: cut to fill one.  One partial round above half: cut into up to eight
// slices where those fill whole rounds 3% better.
size_t gemm_uncut_bytes(uint32_t T, uint32_t slots, int64_t nk, size_t tile)
{
    const uint32_t rem = T % slots;
    uint32_t cut = 0, sk = 0;
    if (T > slots && rem > 0 && rem <= slots / 2 && nk >= 32) {
        cut = rem;
        sk = (uint32_t)std::min<int64_t>(slots / rem, nk / 8);
    } else if (T <= slots / 2 && nk >= 16) {
        cut = T;
        sk = (uint32_t)std::min<int64_t>(slots / T, nk / 4);
    } else if (T <= slots && nk >= 32) {
        double best = (double)T / slots;
        for (uint32_t c = 2; c <= 8 && nk / c >= 8 && T * c <= 2 * slots; c++) {
            const uint32_t items = T * c;
            const double fill = (double)items / (double)((items + slots - 1) / slots * slots);
            if (fill > best * 1.03) {
                best = fill;
                sk = c;
            }
        }
        cut = T;
    }
    if (sk < 2) return 0;
    const int64_t steps = (nk + sk - 1) / sk;
    return (size_t)cut * ((nk + steps - 1) / steps) * tile * sizeof(double);
}

int gemm_device_cus(int *cus) { return device_cus(cus); }

int gemm_reserve_workspace(hipStream_t s)
{
    // Two slots of a tile per run and at most `occ` runs per CU
    // (gemm_split_plan): twice the largest tile (192 x 96) times two runs per
    // CU bounds every request.
    int cus = 0;
    int st = device_cus(&cus);
    if (st != DTCF_OK) return st;
    const size_t tile = std::max<size_t>({128 * 128, 192 * 96, 96 * 192, 2 * 64 * 64, 192 * 64});
    double *ws = nullptr;
    return split_workspace(s, (size_t)cus * 2 * 2 * tile * sizeof(double), SIZE_MAX, &ws);
}

int gemm_f64_launch(GemmArgs g, int cfg, hipStream_t s)
{
    if (g.m <= 0 || g.n <= 0 || g.k <= 0) return DTCF_OK;
    DTCF_REQUIRE((g.m + 63) / 64 * ((g.n + 63) / 64) < (1ll << 31), "gemm: too many tiles");
    switch (cfg) {
    case kCfg128x128: return gemm_tile_128x128(g, s);
    case kCfg192x96: return gemm_tile_192x96(g, s);
    case kCfg96x192: return gemm_tile_96x192(g, s);
    case kCfg64x64: return gemm_tile_64x64(g, s);
    case kCfg192x64: return gemm_tile_192x64(g, s);
    case kCfg64x192: return gemm_tile_64x192(g, s);
    case kCfgThin: {
        const int st = thin_f64_launch(g, s);
        if (st != kThinDecline) return st;
        return gemm_tile_64x64(g, s);
    }
    default: break;
    }
    set_error("gemm: unknown tile configuration");
    return DTCF_ERR_INVALID;
}

}  // namespace dtcf
