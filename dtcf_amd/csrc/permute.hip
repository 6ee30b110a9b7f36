// Strided permute-copy on gfx950: the one kernel behind RRR transpose
// (helper.cc:275-522), the DLTC transpose_<perm> family
// (DLTC/transp-kernel-seq.cc) and the create_big_matrix / revert_big_matrix
// pack and unpack (transpose_helper.cc:149-159, 393-403).
//
// The host folds dims that are adjacent in both input and output, then picks
// two dims for a 2-D tile:
//   q = the dim with the smallest output stride (output-fastest),
//   p = the dim with unit input stride (input-fastest) when it differs from q.
// TRANSPOSE tiles (p != q) go through LDS so that reads run along p and
// writes run along q, both coalesced; straight tiles (q is fastest on both
// sides) copy through registers with lanes along q.  All other dims and the
// tile batch index are decoded once per plane.
#include <algorithm>
#include <type_traits>
#include <vector>

#include "common.hpp"

namespace dtcf {

namespace {

constexpr int kMaxOther = DTCF_MAX_DIMS;

struct PermParams {
    int32_t n_other;
    uint32_t other_ext[kMaxOther];
    FastDiv other_div[kMaxOther];
    int64_t other_istr[kMaxOther];
    int64_t other_ostr[kMaxOther];
    int64_t ext_p, ext_q;
    int64_t istr_p, istr_q, ostr_p, ostr_q;
    uint32_t ntp, ntq;          // tiles along p and q
    FastDiv div_ntq, div_ntp;
    uint64_t per_tile;          // workgroups per batch entry
    uint64_t total;             // total workgroups of work
    int64_t src_step, dst_step;
    double alpha, beta;
};

// 8-byte form, for any extents, offsets and alignment.  A plane is the p x q
// extents at one index of every other dim and batch entry; a work item is
// one Pt x Qt tile of up to `np` consecutive planes, and its threads take its
// elements flat, p fastest to read and q fastest to write (TRANSPOSE, through
// LDS) or q fastest for both.  So short extents fill the waves (tiles of a
// fixed 32 x 32 left 13 of 32 lanes working on a 13 x 47 plane), a plane that
// is contiguous in the output is written in one run, and eight loads per
// thread are in flight.  HBM-bound: 256 tiles of 11 x 13 x 45 x 47, order
// 2,0,3,1: 417 -> 241 us; 12 ns of start-up per workgroup are spread over
// up to 4096 elements.
constexpr int kPlaneElems = 4096;
constexpr int kMaxPlanes = 64;
struct PlaneParams {
    uint32_t Pt, Qt, np;
    FastDiv div_pt, div_qt, div_pq;  // by Pt, Qt, Pt * Qt
    uint64_t planes, items;
    uint32_t others;                 // planes per batch entry
};

template <bool TRANSPOSE>
__global__ __launch_bounds__(256) void permute_kernel(const double *__restrict__ in,
                                                      double *__restrict__ out, PermParams P, PlaneParams L,
                                                      const int64_t *__restrict__ src_off,
                                                      const int64_t *__restrict__ dst_off)
{
    __shared__ double lds[TRANSPOSE ? kPlaneElems : 1];
    __shared__ int64_t soff[kMaxPlanes], doff[kMaxPlanes];
    const uint32_t tid = threadIdx.x, PS = L.Pt | 1, PQ = L.Pt * L.Qt;  // odd LDS pitch
    for (uint64_t it = blockIdx.x; it < L.items; it += gridDim.x) {
        const uint64_t pg = it / ((uint64_t)P.ntp * P.ntq);
        const uint32_t rem = (uint32_t)(it - pg * P.ntp * P.ntq);
        const uint32_t pt = P.div_ntq.div(rem), qt = rem - pt * P.ntq;
        const uint64_t plane0 = pg * L.np;
        const uint32_t np = (uint32_t)min((uint64_t)L.np, L.planes - plane0);
        if (tid < np) {
            const uint64_t t = (plane0 + tid) / L.others;
            uint32_t x = (uint32_t)(plane0 + tid - t * L.others);
            int64_t src = src_off ? src_off[t] : (int64_t)t * P.src_step;
            int64_t dst = dst_off ? dst_off[t] : (int64_t)t * P.dst_step;
            for (int d = P.n_other - 1; d >= 0; d--) {
                const uint32_t q = P.other_div[d].div(x), r = x - q * P.other_ext[d];
                x = q;
                src += (int64_t)r * P.other_istr[d];
                dst += (int64_t)r * P.other_ostr[d];
            }
            const int64_t p0 = (int64_t)pt * L.Pt, q0 = (int64_t)qt * L.Qt;
            soff[tid] = src + p0 * P.istr_p + q0 * P.istr_q;
            doff[tid] = dst + p0 * P.ostr_p + q0 * P.ostr_q;
        }
        __syncthreads();
        const uint32_t pn = (uint32_t)min((int64_t)L.Pt, P.ext_p - (int64_t)pt * L.Pt);
        const uint32_t qn = (uint32_t)min((int64_t)L.Qt, P.ext_q - (int64_t)qt * L.Qt);
        const uint32_t total = np * PQ;
        // element e of the item: plane, and (slow, fast) of its tile
        auto split = [&](uint32_t e, const FastDiv &fast, uint32_t &pl, uint32_t &hi, uint32_t &lo) {
            pl = L.div_pq.div(e);
            const uint32_t r = e - pl * PQ;
            hi = fast.div(r);
            lo = r - hi * fast.d;
        };
        // Elements outside are clamped to one of the item and not stored: loads
        // under a branch wait one by one (368 us where this form takes 257)
        auto locate = [&](uint32_t e, bool p_fast, uint32_t &pl, uint32_t &pp, uint32_t &qq) {
            const uint32_t c = min(e, total - 1);
            if (p_fast) split(c, L.div_pt, pl, qq, pp);
            else split(c, L.div_qt, pl, pp, qq);
            const bool ok = e < total && pp < pn && qq < qn;
            pp = min(pp, pn - 1);
            qq = min(qq, qn - 1);
            return ok;
        };
        auto put = [&](auto count, const double *v, double *const *to, uint32_t ok) {
            constexpr int U = decltype(count)::value;
            if (P.beta == 0.0) {
#pragma unroll
                for (int u = 0; u < U; u++)
                    if (ok >> u & 1) *to[u] = (P.alpha == 1.0) ? v[u] : P.alpha * v[u];
            } else {
                double w[U];
#pragma unroll
                for (int u = 0; u < U; u++) w[u] = *to[u];
#pragma unroll
                for (int u = 0; u < U; u++)
                    if (ok >> u & 1) *to[u] = P.alpha * v[u] + P.beta * w[u];
            }
        };
        // in -> LDS (TRANSPOSE) or out, `U` elements of this thread from e0 on
        auto fetch = [&](auto count, uint32_t e0) {
            constexpr int U = decltype(count)::value;
            double v[U];
            double *to[U];
            uint32_t at[U], ok = 0;
#pragma unroll
            for (int u = 0; u < U; u++) {
                uint32_t pl, pp, qq;
                if (locate(e0 + 256 * u + tid, TRANSPOSE, pl, pp, qq)) ok |= 1u << u;
                if constexpr (TRANSPOSE) at[u] = (pl * L.Qt + qq) * PS + pp;
                else to[u] = out + doff[pl] + (int64_t)qq * P.ostr_q + (int64_t)pp * P.ostr_p;
                v[u] = in[soff[pl] + (int64_t)pp * P.istr_p + (int64_t)qq * P.istr_q];
            }
            if constexpr (TRANSPOSE) {
#pragma unroll
                for (int u = 0; u < U; u++)
                    if (ok >> u & 1) lds[at[u]] = v[u];
            } else {
                put(count, v, to, ok);
            }
        };
        auto store = [&](auto count, uint32_t e0) {  // LDS -> out
            constexpr int U = decltype(count)::value;
            double v[U];
            double *to[U];
            uint32_t ok = 0;
#pragma unroll
            for (int u = 0; u < U; u++) {
                uint32_t pl, pp, qq;
                if (locate(e0 + 256 * u + tid, false, pl, pp, qq)) ok |= 1u << u;
                to[u] = out + doff[pl] + (int64_t)qq * P.ostr_q + (int64_t)pp * P.ostr_p;
                v[u] = lds[(pl * L.Qt + qq) * PS + pp];
            }
            put(count, v, to, ok);
        };
        // eight per thread, fewer for the rest: the clamped ones cost as much
        auto sweep = [&](auto &&step) {
            uint32_t e0 = 0;
            for (; e0 + 1024 < total; e0 += 2048) step(std::integral_constant<int, 8>(), e0);
            if (e0 + 512 < total) step(std::integral_constant<int, 4>(), e0);
            else if (e0 < total) step(std::integral_constant<int, 2>(), e0);
        };
        sweep(fetch);
        __syncthreads();
        if constexpr (TRANSPOSE) {
            sweep(store);
            __syncthreads();
        }
    }
}

// 8-byte TRANSPOSE tile of a fixed 32 x 32, one per workgroup pass, for
// extents that fill it and tensors that the caches hold: eight workgroups per
// CU keep more tiles in flight than the flat form's four, and nothing is
// divided per element.  75 x 2028 (119 MB read and written) 21.0 us, flat
// 30.7; 169 x 169 in 64 tiles 8.9, 10.8.
__global__ __launch_bounds__(256) void permute_tile_kernel(const double *__restrict__ in,
                                                           double *__restrict__ out, PermParams P,
                                                           const int64_t *__restrict__ src_off,
                                                           const int64_t *__restrict__ dst_off)
{
    __shared__ double lds[32][33];
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (uint64_t blk = blockIdx.x; blk < P.total; blk += gridDim.x) {
        const uint64_t t = blk / P.per_tile;
        uint32_t rem = (uint32_t)(blk - t * P.per_tile);
        const uint32_t qt_div = P.div_ntq.div(rem);
        const uint32_t qt = rem - qt_div * P.ntq;
        rem = qt_div;
        const uint32_t pt_div = P.div_ntp.div(rem);
        const uint32_t pt = rem - pt_div * P.ntp;
        rem = pt_div;
        int64_t src = src_off ? src_off[t] : (int64_t)t * P.src_step;
        int64_t dst = dst_off ? dst_off[t] : (int64_t)t * P.dst_step;
        for (int d = P.n_other - 1; d >= 0; d--) {
            const uint32_t q = P.other_div[d].div(rem);
            const uint32_t x = rem - q * P.other_ext[d];
            rem = q;
            src += (int64_t)x * P.other_istr[d];
            dst += (int64_t)x * P.other_ostr[d];
        }
        const int64_t p0 = (int64_t)pt * 32, q0 = (int64_t)qt * 32;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int64_t pp = p0 + tx, qq = q0 + ty + 8 * i;
            if (pp < P.ext_p && qq < P.ext_q)
                lds[ty + 8 * i][tx] = in[src + pp * P.istr_p + qq * P.istr_q];
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int64_t qq = q0 + tx, pp = p0 + ty + 8 * i;
            if (pp < P.ext_p && qq < P.ext_q) {
                double *o = out + dst + qq * P.ostr_q + pp * P.ostr_p;
                const double v = lds[tx][ty + 8 * i];
                if (P.beta == 0.0) *o = (P.alpha == 1.0) ? v : P.alpha * v;
                else *o = P.alpha * v + P.beta * (*o);
            }
        }
        __syncthreads();
    }
}

// 16-byte form of the TRANSPOSE tile, taken when the fast strides are 1 on
// their side, the extents and every other offset even, the buffers 16-byte
// aligned (no per-tile offset tables) and the tile filled to a fifth:
// 64 x 64 through LDS, 16 elements per thread, reads two consecutive p and
// writes two consecutive q per access.  Same values as permute_kernel.
__global__ __launch_bounds__(256) void permute_vec_kernel(const double *__restrict__ in,
                                                          double *__restrict__ out, PermParams P)
{
    constexpr int TP = 64, TQ = 64;
    __shared__ double lds[64][65];
    const int tid = threadIdx.x;
    for (uint64_t blk = blockIdx.x; blk < P.total; blk += gridDim.x) {
        const uint64_t t = blk / P.per_tile;
        uint32_t rem = (uint32_t)(blk - t * P.per_tile);
        const uint32_t qt_div = P.div_ntq.div(rem);
        const uint32_t qt = rem - qt_div * P.ntq;
        rem = qt_div;
        const uint32_t pt_div = P.div_ntp.div(rem);
        const uint32_t pt = rem - pt_div * P.ntp;
        rem = pt_div;
        int64_t src = (int64_t)t * P.src_step, dst = (int64_t)t * P.dst_step;
        for (int d = P.n_other - 1; d >= 0; d--) {
            const uint32_t q = P.other_div[d].div(rem);
            const uint32_t x = rem - q * P.other_ext[d];
            rem = q;
            src += (int64_t)x * P.other_istr[d];
            dst += (int64_t)x * P.other_ostr[d];
        }
        const int64_t p0 = (int64_t)pt * TP, q0 = (int64_t)qt * TQ;
        auto put = [&](double *o, double2 v) {
            if (P.beta == 0.0) {
                if (P.alpha != 1.0) {
                    v.x *= P.alpha;
                    v.y *= P.alpha;
                }
            } else {
                const double2 w = *reinterpret_cast<const double2 *>(o);
                v.x = P.alpha * v.x + P.beta * w.x;
                v.y = P.alpha * v.y + P.beta * w.y;
            }
            *reinterpret_cast<double2 *>(o) = v;
        };
        const int tx = tid & 31, ty = tid >> 5;
        double2 v[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {  // rows q, pairs of p (unit input stride)
            const int64_t pp = p0 + 2 * tx, qq = q0 + ty + 8 * i;
            v[i] = (pp < P.ext_p && qq < P.ext_q)
                       ? *reinterpret_cast<const double2 *>(in + src + pp + qq * P.istr_q)
                       : make_double2(0.0, 0.0);
        }
#pragma unroll
        for (int i = 0; i < 8; i++) {
            lds[ty + 8 * i][2 * tx] = v[i].x;
            lds[ty + 8 * i][2 * tx + 1] = v[i].y;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 8; i++) {  // rows p, pairs of q (unit output stride)
            const int64_t qq = q0 + 2 * tx, pp = p0 + ty + 8 * i;
            if (pp < P.ext_p && qq < P.ext_q)
                put(out + dst + qq + pp * P.ostr_p,
                    make_double2(lds[2 * tx][ty + 8 * i], lds[2 * tx + 1][ty + 8 * i]));
        }
        __syncthreads();
    }
}

struct Dim {
    int64_t ext, istr, ostr;
};

}  // namespace

// Validates and normalises a descriptor: drops unit dims and folds dims that
// are contiguous in both input and output.  Returns the folded dims in
// order of decreasing output stride.
static int fold_dims(const dtcf_strided *d, std::vector<Dim> &dims, bool &empty)
{
    DTCF_REQUIRE(d != nullptr, "permute: null descriptor");
    DTCF_REQUIRE(d->dims >= 1 && d->dims <= DTCF_MAX_DIMS, "permute: dims must be 1..8");
    empty = false;
    std::vector<Dim> v;
    for (int i = 0; i < d->dims; i++) {
        DTCF_REQUIRE(d->ext[i] >= 0, "permute: negative extent");
        if (d->ext[i] == 0) empty = true;
        if (d->ext[i] > 1) v.push_back({d->ext[i], d->istr[i], d->ostr[i]});
    }
    if (v.empty()) v.push_back({1, 1, 1});
    std::stable_sort(v.begin(), v.end(),
                     [](const Dim &a, const Dim &b) { return a.ostr > b.ostr; });
    std::vector<Dim> f;
    for (const Dim &x : v) {
        if (!f.empty()) {
            Dim &b = f.back();
            if (b.istr == x.istr * x.ext && b.ostr == x.ostr * x.ext) {
                b.ext *= x.ext;
                b.istr = x.istr;
                b.ostr = x.ostr;
                continue;
            }
        }
        f.push_back(x);
    }
    dims = f;
    return DTCF_OK;
}

}  // namespace dtcf

using namespace dtcf;

extern "C" int dtcf_permute_copy_f64(const double *in, double *out, const dtcf_strided *desc,
                                     int64_t ntiles, const int64_t *src_off, int64_t src_step,
                                     const int64_t *dst_off, int64_t dst_step, double alpha,
                                     double beta, void *stream)
{
    std::vector<Dim> dims;
    bool empty = false;
    int st = fold_dims(desc, dims, empty);
    if (st != DTCF_OK) return st;
    DTCF_REQUIRE(ntiles >= 0, "permute: negative tile count");
    if (empty || ntiles == 0) return DTCF_OK;
    DTCF_REQUIRE(in != nullptr && out != nullptr, "permute: null buffer");

    // q: output-fastest dim (folded dims are sorted, so it is the last one).
    const int q = (int)dims.size() - 1;
    // p: input-fastest dim if it is a different dim; otherwise the dim with
    // the next smallest output stride.
    int p = -1;
    int64_t best = INT64_MAX;
    for (int i = 0; i < (int)dims.size(); i++)
        if (i != q && dims[i].istr >= 0 && dims[i].istr < best) {
            best = dims[i].istr;
            p = i;
        }
    bool transpose = (p >= 0 && dims[p].istr < dims[q].istr);
    if (!transpose && dims.size() > 1) p = q - 1;

    PermParams P{};
    Dim dq = dims[q];
    Dim dp = p >= 0 ? dims[p] : Dim{1, 0, 0};
    P.ext_p = dp.ext;
    P.ext_q = dq.ext;
    P.istr_p = dp.istr;
    P.ostr_p = dp.ostr;
    P.istr_q = dq.istr;
    P.ostr_q = dq.ostr;
    // 16-byte form: a transpose of unit fast strides, even extents and
    // offsets, aligned buffers, offsets from steps (not tables), whose 64 x 64
    // tiles the extents fill to a fifth at least.  us, 16-byte / flat: 48 x 48
    // 253 / 275, 24 x 48 155 / 162, 32 x 32 150 / 155, below a fifth 24 x 24
    // 225 / 161, 20 x 20 35 / 24, 12 x 48 365 / 253.  (A straight copy gains
    // nothing from it: 64 x 128 199 / 195, 32 x 64 211 / 146.)
    auto fill = [](int64_t ext) { return (double)ext / (double)((ext + 63) / 64 * 64); };
    bool vec = transpose && !src_off && !dst_off && (reinterpret_cast<uintptr_t>(in) & 15) == 0 &&
               (reinterpret_cast<uintptr_t>(out) & 15) == 0 && src_step % 2 == 0 &&
               dst_step % 2 == 0 && dq.ext % 2 == 0 && dq.ostr == 1 && dp.istr == 1 &&
               dp.ext % 2 == 0 && dq.istr % 2 == 0 && dp.ostr % 2 == 0 && fill(dp.ext) * fill(dq.ext) >= 0.2;
    for (int i = 0; vec && i < (int)dims.size(); i++)
        if (i != q && i != p) vec = dims[i].istr % 2 == 0 && dims[i].ostr % 2 == 0;
    // Tiles: 64 x 64 in the 16-byte form; in the flat form at most 64 x 63
    // through LDS (65 x 63 with its odd pitch fills the buffer) or 4096
    // elements straight, the extents cut evenly.
    int64_t TP = 64, TQ = 64;
    PlaneParams L{};
    // The fixed tile: a transpose whose extents fill the 32 x 32 tiles to 0.4
    // at least and do not leave tiles nearly empty past their first (from 40
    // MB on), up to the 256 MB of the last-level cache and a little.  us, fixed
    // / flat: 32 x 13 (36 MB, fill 0.41) 10.2 / 12.7, 19 x 19 (59 MB, 0.35) 17 /
    // 16; 129 x 304 (237 MB) 42.4 / 54.3, 55 x 45 (192 MB, whose second tiles
    // are 0.6 full) 49 / 38; 129 x 63 (329 MB) 83 / 73.
    auto filled = [](int64_t ext) { return (double)ext / (double)((ext + 31) / 32 * 32); };
    auto later = [&](int64_t ext) { return ext <= 32 ? 1.0 : filled(ext); };
    double mb = 16e-6 * (double)ntiles;  // read and written
    for (const Dim &d : dims) mb *= (double)d.ext;
    const bool fixed = transpose && !vec && mb < 275.0 && filled(dp.ext) * filled(dq.ext) >= 0.4 &&
                       (mb < 40.0 || later(dp.ext) * later(dq.ext) >= 0.61);
    if (fixed) {
        TP = TQ = 32;
    } else if (!vec) {
        auto even = [](int64_t ext, int64_t most) {
            const int64_t n = (ext + most - 1) / most;
            return (ext + n - 1) / n;
        };
        // fewer than 1024 tiles of 64 x 63: 32 x 32, so that no CU idles (200
        // of 63 x 65, 15 -> 11 us; one of 1331 x 1177, 13 -> 11)
        uint64_t tiles = (uint64_t)ntiles * ((dp.ext + 63) / 64) * ((dq.ext + 62) / 63);
        for (int i = 0; i < (int)dims.size() && tiles < 1024; i++)
            if (i != q && i != p) tiles *= (uint64_t)dims[i].ext;
        const bool small = tiles < 1024;
        TQ = even(dq.ext, !transpose ? kPlaneElems : small ? 32 : 63);
        TP = even(dp.ext, !transpose ? std::max<int64_t>(1, kPlaneElems / TQ) : small ? 32 : 64);
    }
    const uint64_t ntp = (dp.ext + TP - 1) / TP, ntq = (dq.ext + TQ - 1) / TQ;
    uint64_t per = ntp * ntq;
    int n_other = 0;
    for (int i = 0; i < (int)dims.size(); i++) {
        if (i == q || i == p) continue;
        P.other_ext[n_other] = (uint32_t)dims[i].ext;
        P.other_div[n_other] = FastDiv((uint32_t)dims[i].ext);
        P.other_istr[n_other] = dims[i].istr;
        P.other_ostr[n_other] = dims[i].ostr;
        per *= (uint64_t)dims[i].ext;
        n_other++;
    }
    DTCF_REQUIRE(per < (1ull << 31), "permute: a single tile is too large (> 2^31 workgroups)");
    P.n_other = n_other;
    P.ntp = (uint32_t)ntp;
    P.ntq = (uint32_t)ntq;
    P.div_ntp = FastDiv((uint32_t)ntp);
    P.div_ntq = FastDiv((uint32_t)ntq);
    P.per_tile = per;
    P.total = per * (uint64_t)ntiles;
    P.src_step = src_step;
    P.dst_step = dst_step;
    P.alpha = alpha;
    P.beta = beta;

    const uint64_t max_grid = 256ull * 64;  // plenty of waves in flight per CU
    hipStream_t s = as_stream(stream);
    if (!vec && !fixed) {
        L.Pt = (uint32_t)TP;
        L.Qt = (uint32_t)TQ;
        const uint32_t elems = (transpose ? L.Pt | 1 : L.Pt) * L.Qt;  // at most kPlaneElems
        L.others = (uint32_t)(per / (ntp * ntq));
        L.planes = (uint64_t)L.others * (uint64_t)ntiles;
        L.np = std::max<uint32_t>(1, std::min<uint32_t>(kMaxPlanes, kPlaneElems / elems));
        // small calls: fewer planes per item rather than idle CUs
        while (L.np > 1 && (L.planes + L.np - 1) / L.np * ntp * ntq < 1024) L.np = (L.np + 1) / 2;
        L.items = (L.planes + L.np - 1) / L.np * ntp * ntq;
        L.div_pt = FastDiv(L.Pt);
        L.div_qt = FastDiv(L.Qt);
        L.div_pq = FastDiv(L.Pt * L.Qt);
        const unsigned grid = (unsigned)std::min<uint64_t>(L.items, max_grid);
        if (transpose)
            hipLaunchKernelGGL(permute_kernel<true>, dim3(grid), dim3(256), 0, s, in, out, P, L, src_off, dst_off);
        else
            hipLaunchKernelGGL(permute_kernel<false>, dim3(grid), dim3(256), 0, s, in, out, P, L, src_off, dst_off);
        DTCF_HIP(hipGetLastError());
        return DTCF_OK;
    }
    const unsigned grid = (unsigned)std::min<uint64_t>(P.total, max_grid);
    if (fixed) hipLaunchKernelGGL(permute_tile_kernel, dim3(grid), dim3(256), 0, s, in, out, P, src_off, dst_off);
    else hipLaunchKernelGGL(permute_vec_kernel, dim3(grid), dim3(256), 0, s, in, out, P);
    DTCF_HIP(hipGetLastError());
    return DTCF_OK;
}

// Builds the descriptor for `ntiles` dense row-major tiles of extents w and
// output order out_src (output dim n is input dim out_src[n]).
int dtcf_build_tile_desc(int dims, const int64_t *w, const int32_t *out_src, dtcf_strided *d,
                         int64_t *block)
{
    DTCF_REQUIRE(dims >= 1 && dims <= DTCF_MAX_DIMS, "permute: dims must be 1..8");
    DTCF_REQUIRE(w != nullptr && out_src != nullptr, "permute: null extents or order");
    int seen[DTCF_MAX_DIMS] = {0};
    for (int n = 0; n < dims; n++) {
        DTCF_REQUIRE(out_src[n] >= 0 && out_src[n] < dims && !seen[out_src[n]],
                     "permute: out_src is not a permutation");
        seen[out_src[n]] = 1;
        DTCF_REQUIRE(w[n] >= 0, "permute: negative extent");
    }
    int64_t is[DTCF_MAX_DIMS];
    is[dims - 1] = 1;
    for (int i = dims - 2; i >= 0; i--) is[i] = is[i + 1] * w[i + 1];
    d->dims = dims;
    int64_t os = 1;
    for (int n = dims - 1; n >= 0; n--) {
        d->ext[n] = w[out_src[n]];
        d->istr[n] = is[out_src[n]];
        d->ostr[n] = os;
        os *= d->ext[n];
    }
    *block = os;
    return DTCF_OK;
}

extern "C" int dtcf_permute_tiles_f64(const double *in, double *out, int dims, const int64_t *w,
                                      const int32_t *out_src, int64_t ntiles, void *stream)
{
    dtcf_strided d{};
    int64_t block = 0;
    int st = dtcf_build_tile_desc(dims, w, out_src, &d, &block);
    if (st != DTCF_OK) return st;
    return dtcf_permute_copy_f64(in, out, &d, ntiles, nullptr, block, nullptr, block, 1.0, 0.0,
                                 stream);
}
