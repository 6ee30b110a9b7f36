// The FP64 MFMA tile kernels (v_mfma_f64_16x16x4_f64) and their launch, as
// templates over the C tile; gemm_tile_*.hip instantiate one tile each.
//
// Tiling: a 256-thread workgroup (4 wave64) owns a BM x BN block of C; the
// waves form a (BM/WM) x (BN/WN) grid and each wave owns WM x WN as
// (WM/16) x (WN/16) MFMA 16x16 accumulators (4 doubles per lane each).  K is
// walked in steps of BK = 16 through two LDS stages, one barrier per step,
// the next step loading while this one runs its MFMAs.
//
// LDS layout: 16 rows x 16 k of an operand are two fragments h = 0, 1 of 1
// KiB, 16 bytes per lane l.
//   k pairs (KC: kDK, kVK):   lane l holds row l % 16, k = 8h + 2 (l / 16) + {0, 1}
//   row pairs (kDMN, kVMN):   lane l holds rows 2 (l % 8) + {0, 1} of
//                             k = 8h + 2 ((l / 8) % 4) + l / 32
// The MFMA k-slice (h, t), t = 0, 1, takes k = 8h + 2 fk + t from its four
// lane groups fk = l / 16 in both layouts, so operands of either kind
// combine and the sum over k runs in one order.  A k-pair fragment is read
// with one 16-byte read per lane for both slices, a row-pair one with an
// 8-byte read per slice; every read of a wave is one contiguous span (no
// bank conflicts).
//
// Three ways to fill a stage:
//   direct (both operands' pairs adjacent and 16-byte aligned, no block
//   table): global_load_lds, 16 bytes per lane, lane l's pair straight to
//   byte 16 l of its fragment.  No staging registers and no LDS stores, and
//   the loop body is 64 MFMAs, 16 fragment reads and 8 loads (the register-
//   staged form took 242-256 VGPRs at 128 x 128 and spilled up to 38 for view
//   operands; this one takes 220-240 without spills).  Bound by the FP64
//   MFMA rate: 8192^3 dense 63.7 -> 69.9 TF/s (A m x k, B n x k), 66.4 ->
//   70.3 (B k x n), 2048^3 56.8 -> 61.6; the 9216^3 ring step through its
//   views 65.9 -> 67.3 TF/s.
//   staged (anything else): pairs loaded to registers -- one 16-byte load
//   at 8-byte alignment where the pair is adjacent (every dense operand,
//   whatever its pitch), two 8-byte loads where it is not -- and stored to
//   the other stage after the step's MFMAs are issued.
//   1331 x 1177 x 905, odd pitches: 160 -> 69 us (it ran element loads with
//   bounds checks in every step).
//   table (a view whose block table did not fold): staged, with the blocks'
//   offsets looked up a step ahead and added only when the pair is loaded (an
//   add at the look-up would wait for the data loads issued before it: 64 x
//   64 at 2304^3, both operands in 144 x 144 tiles of a scrambled order, 920
//   us, 567 so; with checked loads in every step 1468).
// Only a K step that is not whole (K % 16), or the last one of a dense
// row-contiguous operand with an odd row count, whose last pair reaches past
// the operand, is loaded element by element with bounds checks (nfast).  Rows past the operand's last (an edge tile) load
// the last row or row pair again: in range, and never stored.
#pragma once
#include <algorithm>
#include <mutex>

#include "common.hpp"
#include "gemm_f64.hpp"
#include "runs.hpp"

namespace dtcf {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));  // 16-byte load at 8-byte alignment

constexpr int BK = 16;
constexpr int NT = 256;
constexpr int KH = BK / 8;  // fragments per 16 rows and K step

// How a kernel fills its stages: through registers, the same with a block
// table on a view operand, straight into LDS.
enum { kStaged = 0, kTable = 1, kDirect = 2 };

template <int MODE>
struct ModeT {
    static constexpr bool KC = (MODE == kDK || MODE == kVK);
    static constexpr bool VIEW = (MODE == kVK || MODE == kVMN);
};

// Element offset of (r, c) in an operand.
template <int MODE>
__device__ inline int64_t op_addr(const OpArgs &o, int64_t r, int64_t c)
{
    if constexpr (MODE == kDK) return r * o.ld + c;
    else if constexpr (MODE == kDMN) return c * o.ld + r;
    else {
        int64_t a = o.rofs[r] + o.cofs[c];
        if (o.blk) {
            const uint32_t rb = o.div_rpb.div((uint32_t)r);
            const uint32_t cb = o.div_cpb.div((uint32_t)c);
            a += o.blk[(int64_t)rb * o.ncb + cb];
        }
        return a;
    }
}

// One wave's share of one operand's stage: P of the ROWS/16 * KH fragments,
// f = wave * P + i: 16-row group f / KH, half f % KH.
template <int ROWS, int MODE, int LOAD>
struct Loader {
    typedef ModeT<MODE> M;
    static constexpr bool DIRECT = LOAD == kDirect, TABLE = LOAD == kTable;
    static constexpr int P = ROWS / 16 * KH / 4;
    static_assert(ROWS % 32 == 0, "whole fragments per wave");
    const double *p0[P];  // row part of the pair (its first row)
    const double *p1[(!DIRECT && !M::KC) ? P : 1];  // second row of a non-adjacent row pair
    int64_t c0[M::VIEW ? P : 1];                    // column offsets of the next step to load
    int64_t c1[(M::VIEW && !DIRECT && M::KC) ? P : 1];
    uint32_t rb[TABLE ? P : 1], rb1[(TABLE && !M::KC) ? P : 1];  // block rows
    int64_t b0[TABLE ? P : 1], b1[TABLE ? P : 1];   // block offsets of the pair's elements
    d2 reg[DIRECT ? 1 : P];

    __device__ static inline int frag_row(int f, int l) { return 16 * (f / KH) + (M::KC ? (l & 15) : 2 * (l & 7)); }
    __device__ static inline int frag_k(int f, int l)
    {
        return 8 * (f % KH) + (M::KC ? 2 * (l >> 4) : 2 * ((l >> 3) & 3) + (l >> 5));
    }

    __device__ inline void init(const OpArgs &o, const double *base, int64_t row0, int64_t rows, int w, int l)
    {
        // whole pairs: rows past the end repeat the last row or row pair (an
        // odd last row is its own pair; nfast keeps its partner in range)
        const int64_t last = M::KC ? rows - 1 : (rows - 1) & ~int64_t(1);
#pragma unroll
        for (int i = 0; i < P; i++) {
            const int f = w * P + i;
            const int64_t r = min(row0 + frag_row(f, l), last);
            if constexpr (MODE == kDK) p0[i] = base + r * o.ld + frag_k(f, l);
            else if constexpr (MODE == kDMN) p0[i] = base + frag_k(f, l) * o.ld + r;
            else {
                p0[i] = base + o.rofs[r];
                if constexpr (!DIRECT && !M::KC) p1[i] = base + o.rofs[min(r + 1, rows - 1)];
                if constexpr (TABLE) {
                    rb[i] = o.div_rpb.div((uint32_t)r);
                    if constexpr (!M::KC) rb1[i] = o.div_rpb.div((uint32_t)min(r + 1, rows - 1));
                }
            }
        }
    }
    // Column and block offsets of K step kt (views): fetched a step before
    // their data, so no data load waits on a table load.
    __device__ inline void fetch(const OpArgs &o, int64_t kt, int w, int l)
    {
        if constexpr (M::VIEW) {
#pragma unroll
            for (int i = 0; i < P; i++) {
                const int64_t c = kt * BK + frag_k(w * P + i, l);
                c0[i] = o.cofs[c];
                if constexpr (!DIRECT && M::KC) c1[i] = o.cofs[c + 1];
                if constexpr (TABLE) {
                    b0[i] = b1[i] = 0;
                    if (!o.blk) continue;  // uniform: the other operand has the table
                    const uint32_t cb = o.div_cpb.div((uint32_t)c);
                    b0[i] = o.blk[rb[i] * o.ncb + cb];
                    if (o.adj) continue;  // uniform: the pair lies in one block
                    if constexpr (M::KC) b1[i] = o.blk[rb[i] * o.ncb + o.div_cpb.div((uint32_t)c + 1)];
                    else b1[i] = o.blk[rb1[i] * o.ncb + cb];
                }
            }
        }
    }
    __device__ inline const double *at(const OpArgs &o, int i, int64_t kt) const
    {
        if constexpr (MODE == kDK) return p0[i] + kt * BK;
        else if constexpr (MODE == kDMN) return p0[i] + kt * BK * o.ld;
        else if constexpr (TABLE) return p0[i] + c0[i] + b0[i];
        else return p0[i] + c0[i];
    }
    // Loads K step kt (kt < nfast) of this wave's fragments: into the stage
    // (direct) or into registers.
    __device__ inline void load(const OpArgs &o, d2 *stage, int64_t kt, int w)
    {
        if constexpr (DIRECT) {
#pragma unroll
            for (int i = 0; i < P; i++)
                __builtin_amdgcn_global_load_lds(
                    (const void *)at(o, i, kt),
                    (__attribute__((address_space(3))) void *)(stage + (w * P + i) * 64), 16, 0, 0);
        } else if (!M::VIEW || o.adj) {  // uniform
#pragma unroll
            for (int i = 0; i < P; i++) reg[i] = *reinterpret_cast<const d2u *>(at(o, i, kt));
        } else if constexpr (M::VIEW) {
#pragma unroll
            for (int i = 0; i < P; i++) {
                reg[i].x = *at(o, i, kt);
                const double *y = M::KC ? p0[i] + c1[M::KC ? i : 0] : p1[M::KC ? 0 : i] + c0[i];
                reg[i].y = TABLE ? y[b1[TABLE ? i : 0]] : *y;
            }
        }
    }
    __device__ inline void store(d2 *stage, int w, int l) const
    {
#pragma unroll
        for (int i = 0; i < (DIRECT ? 0 : P); i++) stage[(w * P + i) * 64 + l] = reg[i];
    }
    __device__ static inline int64_t addr(const OpArgs &o, int64_t r, int64_t c)
    {
        if constexpr (M::VIEW && DIRECT) return o.rofs[r] + o.cofs[c];  // no block table
        else return op_addr<MODE>(o, r, c);
    }
    // Loads and stores one K step element by element, zeros outside.
    __device__ inline void load_checked(const OpArgs &o, const double *base, d2 *stage, int64_t row0,
                                        int64_t rows, int64_t K, int64_t kt, int w, int l) const
    {
#pragma unroll
        for (int i = 0; i < P; i++) {
            const int f = w * P + i;
            const int64_t r = row0 + frag_row(f, l), c = kt * BK + frag_k(f, l);
            const int64_t r1 = M::KC ? r : r + 1, cc1 = M::KC ? c + 1 : c;
            d2 v = {0.0, 0.0};
            if (r < rows && c < K) v.x = base[addr(o, r, c)];
            if (r1 < rows && cc1 < K) v.y = base[addr(o, r1, cc1)];
            stage[f * 64 + l] = v;
        }
    }
};

// Logical tile q -> (tm, tn) through a grouped (8 tile rows) swizzle.
__device__ inline void tile_coords(uint32_t q, uint32_t tiles_m, uint32_t tiles_n, uint32_t &tm,
                                   uint32_t &tn)
{
    const uint32_t GROUP = 8;
    const uint32_t width = GROUP * tiles_n;
    const uint32_t gid = q / width;
    const uint32_t first = gid * GROUP;
    const uint32_t gsz = min(tiles_m - first, GROUP);
    tm = first + (q % width) % gsz;
    tn = (q % width) / gsz;
}

// One workgroup's share of a GEMM: logical tile q over K steps [kt0, kt1);
// a piece of a split tile (split) writes raw sums to workspace slot sidx.
template <int BM, int BN, int WM, int WN, int AMODE, int BMODE, int LOAD>
__device__ __forceinline__ void gemm_tile(const GemmArgs &g, uint32_t q, int64_t kt0, int64_t kt1,
                                          bool split, uint32_t sidx)
{
    static_assert((BM / WM) * (BN / WN) == 4, "four waves per workgroup");
    constexpr bool DIRECT = LOAD == kDirect;
    constexpr int FM = WM / 16, FN = WN / 16;
    constexpr int FA = BM / 16 * KH, FB = BN / 16 * KH;  // fragments per stage
    constexpr bool AKC = ModeT<AMODE>::KC, BKC = ModeT<BMODE>::KC;
    extern __shared__ d2 smem[];  // two stages of (FA + FB) x 64

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / (BN / WN), wn = wave % (BN / WN);

    uint32_t tm, tn;
    tile_coords(q, g.tiles_m, g.tiles_n, tm, tn);
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;

    Loader<BM, AMODE, LOAD> la;
    Loader<BN, BMODE, LOAD> lb;
    d4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) acc[i][j] = (d4){0.0, 0.0, 0.0, 0.0};

    // K steps [0, n) of this share; the first nf are loaded unchecked.
    const int n = (int)(kt1 - kt0), nf = (int)min(max(g.nfast - kt0, int64_t(0)), kt1 - kt0);
    auto stage = [&](int s) __attribute__((always_inline)) { return smem + (s & 1) * (FA + FB) * 64; };
    auto begin = [&](int s) __attribute__((always_inline)) {
        la.load(g.a, stage(s), kt0 + s, wave);
        lb.load(g.b, stage(s) + FA * 64, kt0 + s, wave);
        if (s + 1 < nf) {
            la.fetch(g.a, kt0 + s + 1, wave, lane);
            lb.fetch(g.b, kt0 + s + 1, wave, lane);
        }
    };
    auto finish = [&](int s) __attribute__((always_inline)) {
        la.store(stage(s), wave, lane);
        lb.store(stage(s) + FA * 64, wave, lane);
    };
    auto checked = [&](int s) __attribute__((always_inline)) {
        la.load_checked(g.a, g.A, stage(s), m0, g.m, g.k, kt0 + s, wave, lane);
        lb.load_checked(g.b, g.B, stage(s) + FA * 64, n0, g.n, g.k, kt0 + s, wave, lane);
    };
    // The direct loads are counted by vmcnt and the compiler does not tie
    // them to the LDS reads: every wave waits for its own, then the barrier
    // makes everyone's visible.  The clobber keeps LDS accesses on their side;
    // the scheduling barrier keeps the step's MFMAs above the wait (the
    // compiler otherwise sinks them below it, and a step then starts by
    // waiting for the loads it just issued: 25.4 instead of 23.6 ms for the
    // ring step).
    auto sync = []() __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(7 << 4);  // vmcnt 0, lgkmcnt 0
        asm volatile("s_barrier" ::: "memory");
    };
    // The second half's fragments are read after the first MFMAs of the
    // first half are issued, and complete under the rest of them.
    auto compute = [&](int s, bool store_next) __attribute__((always_inline)) {
        const d2 *a_s = stage(s), *b_s = a_s + FA * 64;
        d2 af[KH][FM], bf[KH][FN];
        auto frags = [&](int h) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < FN; j++) {
                const d2 *f = b_s + ((wn * FN + j) * KH + h) * 64;
                const double *e = reinterpret_cast<const double *>(f);
                if constexpr (BKC) bf[h][j] = f[lane];
                else bf[h][j] = (d2){e[lane], e[64 + lane]};
            }
#pragma unroll
            for (int i = 0; i < FM; i++) {
                const d2 *f = a_s + ((wm * FM + i) * KH + h) * 64;
                const double *e = reinterpret_cast<const double *>(f);
                if constexpr (AKC) af[h][i] = f[lane];
                else af[h][i] = (d2){e[lane], e[64 + lane]};
            }
        };
        auto row = [&](int h, int t, int i) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < FN; j++)
                acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[h][i][t], bf[h][j][t], acc[i][j], 0, 0, 0);
        };
        // The wave starting a K step takes issue priority for its first half,
        // so the two workgroups sharing a CU drift apart and one's loads and
        // barrier overlap the other's MFMAs.
        __builtin_amdgcn_s_setprio(1);
        frags(0);
        __builtin_amdgcn_sched_barrier(0);
        row(0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        frags(1);
#pragma unroll
        for (int x = 1; x < 2 * FM; x++) row(0, x / FM, x % FM);
        __builtin_amdgcn_s_setprio(0);
#pragma unroll
        for (int x = 0; x < 2 * FM; x++) row(1, x / FM, x % FM);
        // The other stage was last read before the previous barrier: the
        // staged form stores the next step after the last MFMAs are issued.
        if (!DIRECT && store_next) finish(s + 1);
    };

    int s = -1;
    if (nf > 0) {
        la.init(g.a, g.A, m0, g.m, wave, lane);
        lb.init(g.b, g.B, n0, g.n, wave, lane);
        la.fetch(g.a, kt0, wave, lane);
        lb.fetch(g.b, kt0, wave, lane);
        begin(0);
        finish(0);
        sync();
        for (s = 0; s + 1 < nf; s++) {
            begin(s + 1);
            compute(s, true);
            sync();
        }
    }
    // the last unchecked step and the checked one, out of the loop's code
    for (; s < n; s++) {
        if (s + 1 < n) checked(s + 1);
        if (s >= 0) compute(s, false);
        sync();
    }

    const int fr = lane & 15, fq = lane >> 4;
    if (split) {
        // raw sums to the workspace, [slot][BM][BN]; the reduce kernel adds
        // the tile's pieces to C
        double *w = g.ws + (int64_t)sidx * BM * BN;
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    w[(wm * WM + i * 16 + fq + 4 * r) * BN + wn * WN + j * 16 + fr] = acc[i][j][r];
        return;
    }

    // Epilogue: C += alpha * acc  (beta = 1, as every reference call site),
    // or C = alpha * acc when the caller asked for an overwrite.  Sixteen
    // rows at a time: their addresses, then the old values in one batch of
    // loads, then the stores (a load per store would wait for each in turn).
    const double alpha = g.alpha;
    int64_t co[FN];
#pragma unroll
    for (int j = 0; j < FN; j++) {
        const int64_t col = min(n0 + wn * WN + j * 16 + fr, g.n - 1);
        co[j] = g.cview ? g.c.cofs[col] : col;
    }
#pragma unroll
    for (int i = 0; i < FM; i++) {
        int64_t ad[4][FN];
        double old[4][FN];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int64_t row = min(m0 + wm * WM + i * 16 + fq + 4 * r, g.m - 1);
            const int64_t ro = g.cview ? g.c.rofs[row] : row * g.c.ld;
#pragma unroll
            for (int j = 0; j < FN; j++) {
                ad[r][j] = ro + co[j];
                if (g.cview && g.c.blk) {
                    const int64_t col = min(n0 + wn * WN + j * 16 + fr, g.n - 1);
                    ad[r][j] += g.c.blk[(int64_t)g.c.div_rpb.div((uint32_t)row) * g.c.ncb +
                                        g.c.div_cpb.div((uint32_t)col)];
                }
            }
        }
        if (!g.overwrite) {
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int j = 0; j < FN; j++) old[r][j] = g.C[ad[r][j]];
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            if (m0 + wm * WM + i * 16 + fq + 4 * r >= g.m) continue;
#pragma unroll
            for (int j = 0; j < FN; j++) {
                if (n0 + wn * WN + j * 16 + fr >= g.n) continue;
                const double v = alpha * acc[i][j][r];
                g.C[ad[r][j]] = g.overwrite ? v : old[r][j] + v;
            }
        }
    }
}

// K steps that need no bounds checks (gemm_tile): whole ones, less the last
// when a row pair of a dense row-contiguous operand with an odd row count
// reads one element past the operand's last k row.
inline int64_t fast_steps(int64_t k, bool odd_pairs)
{
    return (odd_pairs && k % BK == 0) ? k / BK - 1 : k / BK;
}

// Workgroups per CU: two of the large tiles (their LDS stages take 64-74
// KiB each), four of 64 x 64 (32 KiB, 128 VGPRs).
template <int BM, int BN>
struct Occ {
    static constexpr int v = BM * BN <= 64 * 64 ? 4 : 2;
};

template <int BM, int BN, int WM, int WN, int AMODE, int BMODE, int LOAD>
__global__ __launch_bounds__(NT, (Occ<BM, BN>::v)) void gemm_f64_kernel(GemmArgs g)
{
    // Workgroups below t_full own whole tiles; their ids are first remapped
    // so consecutive tiles land on one XCD (its own L2).  Workgroups above
    // own one run of the split tiles' K steps each.
    const uint32_t bid = blockIdx.x;
    const int64_t nk = (g.k + BK - 1) / BK;
    uint32_t q, slot = 0;
    int64_t k0 = 0, left = nk;
    if (bid < g.t_full) {
        q = bid;
        if ((g.t_full & 7u) == 0) q = (bid & 7u) * (g.t_full >> 3) + (bid >> 3);
    } else {
        const uint32_t w = run_index(bid - g.t_full, g.sw);
        const int64_t s = run_begin(w, g.sw, g.steps), t = div_small(s, nk);
        left = run_begin(w + 1, g.sw, g.steps) - s;
        q = g.t_full + (uint32_t)t;
        k0 = s - t * nk;
        slot = 2 * w;
    }
    for (; left > 0; q++) {
        const int64_t k1 = min(nk, k0 + left);
        gemm_tile<BM, BN, WM, WN, AMODE, BMODE, LOAD>(g, q, k0, k1, k0 > 0 || k1 < nk, slot);
        left -= k1 - k0;
        k0 = 0;
        slot |= 1;
    }
}

// Index of the last entry not above x (GemmGroupArgs).
template <typename U>
__device__ inline int group_problem(const U (&first)[kGroupMax], U x)
{
    int p = 0;
#pragma unroll
    for (int i = 1; i < kGroupMax; i++) p = x >= first[i] ? i : p;
    return p;
}

// Several independent dense GEMMs C_p (+)= alpha A_p B_p^T in one launch.
// Problem p's whole tiles own workgroups [wg0_p, wg0_p + t_whole_p); every
// eighth of them, one XCD's, takes a contiguous part of the problem's tile
// order, as in a lone launch.  (Cutting the list of all whole tiles into eight
// runs of equal work, one per XCD, was measured slower: 8 x 2048^3 55.0
// against 56.6 TF/s, 2 x 4096 x 4096 x 2048 59.0 against 63.7.  Rounding each
// problem up to whole rounds of XCDs leaves workgroups that exit at once, and
// the chip then fills unevenly: 222 tiles of 128 x 128 x 630 in eight problems
// 167 us, 108 without; 1004 tiles of 128 x 128 x 1380 897, 705.)  The
// workgroups after wg_whole each own one run of the split tiles' K steps.
template <int BM, int BN, int WM, int WN, int AM, int BMD, int LOAD>
__global__ __launch_bounds__(NT, (Occ<BM, BN>::v)) void gemm_f64_group_kernel(GemmGroupArgs ga)
{
    const uint32_t bid = blockIdx.x;
    int p = 0;
    uint32_t q = 0, w = 0;
    int64_t s = 0, e = 1;
    const bool whole = bid < ga.wg_whole;
    if (whole) {
        p = group_problem(ga.wg0, bid);
        const GemmGroupProb &P = ga.p[p];
        const uint32_t local = bid - ga.wg0[p], x = local & 7u;
        q = x * (P.t_whole >> 3) + min(x, P.t_whole & 7u) + (local >> 3);
    } else {
        w = run_index(bid - ga.wg_whole, ga.sw);
        s = run_begin(w, ga.sw, ga.steps);
        e = run_begin(w + 1, ga.sw, ga.steps);
    }
    for (uint32_t seg = 0; s < e; seg = 1) {
        int64_t k0 = 0, k1;
        if (!whole) p = group_problem(ga.step0, s);
        const GemmGroupProb &P = ga.p[p];
        const int64_t nk = (P.k + BK - 1) / BK;
        if (whole) {
            k1 = nk;
            s = e;
        } else {
            const int64_t t = div_small(s - ga.step0[p], nk);
            q = P.t_whole + (uint32_t)t;
            k0 = s - ga.step0[p] - t * nk;
            k1 = min(nk, k0 + (e - s));
            s += k1 - k0;
        }
        GemmArgs g{};
        g.m = P.m;
        g.n = P.n;
        g.k = P.k;
        g.nfast = P.nfast;
        g.alpha = ga.alpha;
        g.A = P.A;
        g.B = P.B;
        g.C = P.C;
        g.a.ld = P.lda;
        g.b.ld = P.ldb;
        g.c.ld = P.ldc;
        g.tiles_m = P.tiles_m;
        g.tiles_n = P.tiles_n;
        g.overwrite = ga.overwrite;
        g.ws = ga.ws;
        gemm_tile<BM, BN, WM, WN, AM, BMD, LOAD>(g, q, k0, k1, k0 > 0 || k1 < nk, 2 * w + seg);
    }
}

__device__ inline void put_sum(const GemmArgs &g, int64_t row, int64_t col, double sum)
{
    const int64_t addr = g.cview ? op_addr<kVK>(g.c, row, col) : row * g.c.ld + col;
    if (g.overwrite) g.C[addr] = g.alpha * sum;
    else g.C[addr] += g.alpha * sum;
}

// Adds alpha times the pieces of each split tile to (or, overwriting, stores
// them in) C.
template <int BM, int BN>
__global__ __launch_bounds__(256) void split_reduce_kernel(GemmArgs g)
{
    const uint32_t t = blockIdx.y;  // split tile
    uint32_t tm, tn;
    tile_coords(g.t_full + t, g.tiles_m, g.tiles_n, tm, tn);
    const int64_t nk = (g.k + BK - 1) / BK;
    const int e = blockIdx.x * 256 + threadIdx.x;
    const int64_t row = (int64_t)tm * BM + e / BN, col = (int64_t)tn * BN + e % BN;
    if (row >= g.m || col >= g.n) return;
    bool whole;
    const double sum = sum_pieces(g.ws, t, gridDim.y, nk, g.sw, g.steps, BM * BN, e, whole);
    if (!whole) put_sum(g, row, col, sum);
}

// The same over a group.
template <int BM, int BN>
__global__ __launch_bounds__(256) void group_split_reduce_kernel(GemmGroupArgs ga)
{
    const int p = group_problem(ga.tail0, blockIdx.y);
    const GemmGroupProb &P = ga.p[p];
    const uint32_t t = blockIdx.y - ga.tail0[p];  // split tile of the problem
    uint32_t tm, tn;
    tile_coords(P.t_whole + t, P.tiles_m, P.tiles_n, tm, tn);
    const int64_t nk = (P.k + BK - 1) / BK;
    const int e = blockIdx.x * 256 + threadIdx.x;
    const int64_t row = (int64_t)tm * BM + e / BN, col = (int64_t)tn * BN + e % BN;
    if (row >= P.m || col >= P.n) return;
    bool whole;
    const double sum = sum_runs(ga.ws, ga.step0[p] + t * nk, nk, ga.sw, ga.steps, BM * BN, e, whole);
    if (whole) return;
    GemmArgs g{};
    g.C = P.C;
    g.c.ld = P.ldc;
    g.alpha = ga.alpha;
    g.overwrite = ga.overwrite;
    put_sum(g, row, col, sum);
}

// Large dynamic LDS needs the attribute once per kernel.
template <typename K>
int allow_lds(K kern, size_t lds, std::once_flag &once, hipError_t &err)
{
    if (lds > 65536)
        std::call_once(once, [&] {
            err = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        });
    DTCF_HIP(err);
    return DTCF_OK;
}

// gemm_uncut_bytes of a product on the tiles that its shape alone would take,
// two workgroups per CU.
inline size_t uncut_bytes(const GemmArgs &g, int cus)
{
    const int cfg = pick_config(g.m, g.n, g.k, true);
    const TileRate t = tile_rate(cfg == kCfgThin ? kCfg64x64 : cfg);
    const int64_t T = ((g.m + t.bm - 1) / t.bm) * ((g.n + t.bn - 1) / t.bn);
    return gemm_uncut_bytes((uint32_t)T, 2 * cus, (g.k + BK - 1) / BK, (size_t)t.bm * t.bn);
}

template <int CFG, int BM, int BN, int WM, int WN, int AM, int BMD, int LOAD>
int launch_one(GemmArgs g, hipStream_t s)
{
    auto kern = gemm_f64_kernel<BM, BN, WM, WN, AM, BMD, LOAD>;
    constexpr size_t lds = (size_t)2 * (BM + BN) * BK * sizeof(double);
    static std::once_flag once;
    static hipError_t attr_err = hipSuccess;
    int st = allow_lds(kern, lds, once, attr_err);
    if (st != DTCF_OK) return st;
    int cus = 0;
    st = gemm_device_cus(&cus);
    if (st != DTCF_OK) return st;
    const uint32_t T = g.tiles_m * g.tiles_n;
    const int64_t nk = (g.k + BK - 1) / BK;
    SplitPlan sp = gemm_split_plan(T, nk, (int64_t)g.tiles_m * BM + (int64_t)g.tiles_n * BN, cus,
                                   tile_rate(CFG, g.a.gather || g.b.gather));
    if (sp.nsplit) {
        st = gemm_workspace(s, (size_t)2 * sp.sw * BM * BN * sizeof(double), &g.ws, uncut_bytes(g, cus));
        if (st != DTCF_OK) return st;
        if (!g.ws) sp = SplitPlan();
    }
    g.t_full = T - sp.nsplit;
    g.sw = sp.sw;
    g.steps = (int64_t)sp.nsplit * nk;
    hipLaunchKernelGGL(kern, dim3(g.t_full + g.sw), dim3(NT), lds, s, g);
    DTCF_HIP(hipGetLastError());
    if (sp.nsplit) {
        hipLaunchKernelGGL((split_reduce_kernel<BM, BN>), dim3(BM * BN / 256, sp.nsplit), dim3(256), 0, s, g);
        DTCF_HIP(hipGetLastError());
    }
    return DTCF_OK;
}

template <int CFG, int BM, int BN, int WM, int WN, int LOAD>
int launch_modes(const GemmArgs &g, hipStream_t s)
{
    const int am = g.amode, bm = g.bmode;
    if constexpr (LOAD != kTable) {
        if (am == kDK && bm == kDK) return launch_one<CFG, BM, BN, WM, WN, kDK, kDK, LOAD>(g, s);
        if (am == kDK && bm == kDMN) return launch_one<CFG, BM, BN, WM, WN, kDK, kDMN, LOAD>(g, s);
        if (am == kDMN && bm == kDK) return launch_one<CFG, BM, BN, WM, WN, kDMN, kDK, LOAD>(g, s);
        if (am == kDMN && bm == kDMN) return launch_one<CFG, BM, BN, WM, WN, kDMN, kDMN, LOAD>(g, s);
    }
    if (am == kVK && bm == kVK) return launch_one<CFG, BM, BN, WM, WN, kVK, kVK, LOAD>(g, s);
    if (am == kVK && bm == kVMN) return launch_one<CFG, BM, BN, WM, WN, kVK, kVMN, LOAD>(g, s);
    if (am == kVMN && bm == kVK) return launch_one<CFG, BM, BN, WM, WN, kVMN, kVK, LOAD>(g, s);
    if (am == kVMN && bm == kVMN) return launch_one<CFG, BM, BN, WM, WN, kVMN, kVMN, LOAD>(g, s);
    set_error("gemm: unsupported operand mode combination");
    return DTCF_ERR_INVALID;
}

template <int CFG, int BM, int BN, int WM, int WN>
int launch_tile(GemmArgs g, hipStream_t s)
{
    g.tiles_m = (uint32_t)((g.m + BM - 1) / BM);
    g.tiles_n = (uint32_t)((g.n + BN - 1) / BN);
    g.nfast = fast_steps(g.k, (g.amode == kDMN && g.m % 2) || (g.bmode == kDMN && g.n % 2));
    // direct loads need every pair adjacent and 16-byte aligned
    if (g.a.vec2 && g.b.vec2) return launch_modes<CFG, BM, BN, WM, WN, kDirect>(g, s);
    if ((g.amode >= kVK && g.a.blk) || (g.bmode >= kVK && g.b.blk))
        return launch_modes<CFG, BM, BN, WM, WN, kTable>(g, s);
    return launch_modes<CFG, BM, BN, WM, WN, kStaged>(g, s);
}

template <int CFG, int BM, int BN, int WM, int WN, int AM, int BMD, int LOAD>
int launch_group(GemmGroupArgs ga, hipStream_t s)
{
    auto kern = gemm_f64_group_kernel<BM, BN, WM, WN, AM, BMD, LOAD>;
    constexpr size_t lds = (size_t)2 * (BM + BN) * BK * sizeof(double);
    static std::once_flag once;
    static hipError_t attr_err = hipSuccess;
    int st = allow_lds(kern, lds, once, attr_err);
    if (st != DTCF_OK) return st;
    uint64_t total = 0;
    int64_t steps = 0, nk_min = INT64_MAX;
    for (int i = 0; i < ga.np; i++) {
        GemmGroupProb &P = ga.p[i];
        nk_min = std::min<int64_t>(nk_min, (P.k + BK - 1) / BK);
        P.tiles_m = (uint32_t)((P.m + BM - 1) / BM);
        P.tiles_n = (uint32_t)((P.n + BN - 1) / BN);
        P.nfast = fast_steps(P.k, (AM == kDMN && P.m % 2) || (BMD == kDMN && P.n % 2));
        total += (uint64_t)P.tiles_m * P.tiles_n;
        steps += (int64_t)P.tiles_m * P.tiles_n * ((P.k + BK - 1) / BK);
    }
    DTCF_REQUIRE(total + 8 * kGroupMax < (1ull << 31), "gemm group: too many tiles");
    if (total == 0) return DTCF_OK;
    // The split is planned for the group's mean K and taken from the last
    // problems (the shortest in K).
    int cus = 0;
    st = gemm_device_cus(&cus);
    if (st != DTCF_OK) return st;
    // Past one round of 64 x 64 tiles a cut has to gain more: four workgroups
    // per CU absorb the ragged end of problems of different K, which equal runs
    // then lengthen by 10 to 30 us (1802 tiles x 930: 237 us whole, 265-270 cut;
    // 1354 x 800: 158, 171; 1568 x 850: 195, 218; but 8525 x 2050: 2160, 2132).
    TileRate rate = tile_rate(CFG);
    if (Occ<BM, BN>::v == 4 && total > (uint64_t)cus * 4) rate.cut_us += 20.0;
    SplitPlan sp = gemm_split_plan((uint32_t)total, std::max<int64_t>(1, steps / (int64_t)total), 0, cus, rate);
    ga.ws = nullptr;
    if (sp.nsplit) {
        st = gemm_workspace(s, (size_t)2 * sp.sw * BM * BN * sizeof(double), &ga.ws,
                            gemm_uncut_bytes((uint32_t)total, 2 * cus, nk_min, (size_t)BM * BN));
        if (st != DTCF_OK) return st;
        if (!ga.ws) sp = SplitPlan();
    }
    uint32_t left = sp.nsplit;
    for (int i = ga.np - 1; i >= 0; i--) {
        GemmGroupProb &P = ga.p[i];
        const uint32_t T = P.tiles_m * P.tiles_n, take = std::min(left, T);
        P.t_whole = T - take;
        left -= take;
    }
    uint64_t wg = 0;
    uint32_t tail = 0;
    ga.steps = 0;
    for (int i = 0; i < kGroupMax; i++) {
        if (i >= ga.np) {
            ga.wg0[i] = ga.tail0[i] = UINT32_MAX;
            ga.step0[i] = INT64_MAX;
            continue;
        }
        const GemmGroupProb &P = ga.p[i];
        ga.wg0[i] = (uint32_t)wg;
        wg += P.t_whole;
        ga.tail0[i] = tail;
        ga.step0[i] = ga.steps;
        const uint32_t cut = P.tiles_m * P.tiles_n - P.t_whole;
        tail += cut;
        ga.steps += cut * ((P.k + BK - 1) / BK);
    }
    ga.wg_whole = (uint32_t)wg;
    ga.sw = (uint32_t)std::min<int64_t>(sp.sw, ga.steps);
    hipLaunchKernelGGL(kern, dim3(ga.wg_whole + ga.sw), dim3(NT), lds, s, ga);
    DTCF_HIP(hipGetLastError());
    if (ga.sw) {
        hipLaunchKernelGGL((group_split_reduce_kernel<BM, BN>), dim3(BM * BN / 256, sp.nsplit), dim3(256), 0, s, ga);
        DTCF_HIP(hipGetLastError());
    }
    return DTCF_OK;
}

template <int CFG, int BM, int BN, int WM, int WN, int LOAD>
int launch_group_modes(const GemmGroupArgs &ga, int amode, int bmode, hipStream_t s)
{
    if (amode == kDK && bmode == kDK) return launch_group<CFG, BM, BN, WM, WN, kDK, kDK, LOAD>(ga, s);
    if (amode == kDK && bmode == kDMN) return launch_group<CFG, BM, BN, WM, WN, kDK, kDMN, LOAD>(ga, s);
    if (amode == kDMN && bmode == kDK) return launch_group<CFG, BM, BN, WM, WN, kDMN, kDK, LOAD>(ga, s);
    if (amode == kDMN && bmode == kDMN) return launch_group<CFG, BM, BN, WM, WN, kDMN, kDMN, LOAD>(ga, s);
    set_error("gemm group: unsupported operand layout");
    return DTCF_ERR_INVALID;
}

template <int CFG, int BM, int BN, int WM, int WN>
int launch_group_tile(const GemmGroupArgs &ga, int amode, int bmode, hipStream_t s)
{
    bool direct = true;
    for (int i = 0; i < ga.np; i++) direct = direct && ga.p[i].vec2a && ga.p[i].vec2b;
    if (direct) return launch_group_modes<CFG, BM, BN, WM, WN, kDirect>(ga, amode, bmode, s);
    return launch_group_modes<CFG, BM, BN, WM, WN, kStaged>(ga, amode, bmode, s);
}

}  // namespace
}  // namespace dtcf
