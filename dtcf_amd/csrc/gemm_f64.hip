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

// CU count per device, and the tail-split workspace per (device, stream):
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

int split_workspace(hipStream_t s, size_t need, double **ws)
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

// How many of T tiles to cut into K slices (nsplit, the last ones) and
// into how many (sk >= 2; sk < 2 means no split), for `slots` resident
// workgroups and nk K steps per tile.  A last partial round of at most half
// the slots: its tiles are cut to fill one round.  Under-filled grid (at
// most half the slots): every tile is cut.  One partial round (more than
// half the slots, at most all): every tile is cut into the sk <= 8 slices
// that fill whole rounds best, within two rounds of slots, when that beats
// the unsplit fill by 3% (a 340-tile GEMM on 512 slots: 3 slices, 1020
// items in 2 rounds, 66% -> 99.6% of the slots busy).  In every case
// nsplit * sk <= 2 * slots, and every slice is non-empty.
void gemm_tail_split(uint32_t T, uint32_t slots, int64_t nk, uint32_t &nsplit, uint32_t &sk)
{
    const uint32_t rem = T % slots;
    nsplit = 0;
    sk = 0;
    if (T > slots && rem > 0 && rem <= slots / 2 && nk >= 32) {
        nsplit = rem;
        sk = std::min<uint32_t>(slots / rem, (uint32_t)(nk / 8));
    } else if (T <= slots / 2 && nk >= 16) {
        nsplit = T;
        sk = std::min<uint32_t>(slots / T, (uint32_t)(nk / 4));
    } else if (T <= slots && nk >= 32) {
        double best = (double)T / slots;
        for (uint32_t c = 2; c <= 8 && nk / c >= 8 && T * c <= 2 * slots; c++) {
            const uint32_t items = T * c;
            const double fill = (double)items / (double)(((items + slots - 1) / slots) * slots);
            if (fill > best * 1.03) {
                best = fill;
                sk = c;
            }
        }
        if (sk >= 2) nsplit = T;
    }
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

int gemm_workspace(hipStream_t s, size_t need, double **ws) { return split_workspace(s, need, ws); }

int gemm_device_cus(int *cus) { return device_cus(cus); }

int gemm_reserve_workspace(hipStream_t s)
{
    // nsplit * sk <= 2 * slots for every configuration, and slots <= 2 per
    // CU for the tiles that split (Occ), so twice the largest tile area
    // times two slots per CU bounds every request.
    int cus = 0;
    int st = device_cus(&cus);
    if (st != DTCF_OK) return st;
    const size_t tile = std::max<size_t>({128 * 128, 192 * 96, 96 * 192, 64 * 64, 192 * 64});
    double *ws = nullptr;
    return split_workspace(s, (size_t)cus * 2 * 2 * tile * sizeof(double), &ws);
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
