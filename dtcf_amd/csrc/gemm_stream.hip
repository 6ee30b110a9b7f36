// Streaming kernels for the FP64 GEMM shapes the C tiles serve badly:
// matrix-vector products (gemv_kernel, gemv_rows_kernel) and thin products
// with one side at most 48 (192 with short K) and short K (thin_kernel).
// Each is bound by streaming its long operand from HBM.
#include <algorithm>
#include <mutex>

#include "common.hpp"
#include "gemm_tile.hpp"

namespace dtcf {
namespace {

// Matrix-vector product (GemvArgs): the product is HBM-bound (every element
// of M is used once), so instead of MFMA tiles that would run 63 of 64
// columns on padding, each wave takes one row at a time, its lanes read
// 16-byte column pairs 128 columns apart (eight loads in flight per lane),
// x sits in LDS, and the wave sums its lanes in a fixed tree: the order of
// the additions does not depend on timing.
__global__ __launch_bounds__(256) void gemv_kernel(GemvArgs g)
{
    extern __shared__ double xs[];
    for (int64_t c = threadIdx.x; c < g.k; c += 256) xs[c] = g.X[op_addr<kVK>(g.xv, 0, c)];
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int64_t nw = (int64_t)gridDim.x * 4;
    for (int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); r < g.rows; r += nw) {
        const double *row = g.M + g.mrofs[r];
        double acc[8];
#pragma unroll
        for (int u = 0; u < 8; u++) acc[u] = 0.0;
        int64_t c = 2 * lane;
        for (; c + 7 * 128 < g.k; c += 8 * 128) {
            d2 a[8];
#pragma unroll
            for (int u = 0; u < 8; u++) a[u] = *(const d2 *)(row + g.mcofs[c + u * 128]);
#pragma unroll
            for (int u = 0; u < 8; u++) {
                acc[u] = fma(a[u].x, xs[c + u * 128], acc[u]);
                acc[u] = fma(a[u].y, xs[c + u * 128 + 1], acc[u]);
            }
        }
        for (int u = 0; c < g.k; c += 128, u++) {
            const d2 a = *(const d2 *)(row + g.mcofs[c]);
            acc[u] = fma(a.x, xs[c], acc[u]);
            acc[u] = fma(a.y, xs[c + 1], acc[u]);
        }
        double v = ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7]));
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
        if (lane == 0) {
            int64_t addr;
            if (g.yview) addr = g.ycol ? op_addr<kVK>(g.yv, r, 0) : op_addr<kVK>(g.yv, 0, r);
            else addr = g.ycol ? r * g.ldy : r;
            if (g.overwrite) g.Y[addr] = g.alpha * v;
            else g.Y[addr] += g.alpha * v;
        }
    }
}

// Matrix-vector product with M's row pairs adjacent (GemvArgs, mrofs of
// even rows point at pairs): each lane owns a pair of rows and streams one
// 16-byte load per column, the column offset and x(c) being the same for
// the whole wave (scalar loads); a workgroup's 16 waves take 64 row pairs
// each over their own sixteenth of the workgroup's columns, in column
// order, and the sixteen partial sums are added in wave order through LDS.
// With few rows the columns are also split over gridDim.y workgroups, whose
// partial sums (ws[slice][row]) gemv_rows_reduce adds in slice order: the
// order of the additions never depends on timing.
constexpr int kGemvRowsWaves = 16;
__device__ inline void gemv_store(const GemvArgs &g, int64_t r, double v)
{
    int64_t addr;
    if (g.yview) addr = g.ycol ? op_addr<kVK>(g.yv, r, 0) : op_addr<kVK>(g.yv, 0, r);
    else addr = g.ycol ? r * g.ldy : r;
    if (g.overwrite) g.Y[addr] = v;
    else g.Y[addr] += v;
}

__global__ __launch_bounds__(64 * kGemvRowsWaves) void gemv_rows_kernel(GemvArgs g, double *ws)
{
    __shared__ d2 red[kGemvRowsWaves][64];
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t npairs = g.rows / 2;
    const int64_t pr = (int64_t)blockIdx.x * 64 + lane;
    const double *row = g.M + g.mrofs[2 * min(pr, npairs - 1)];
    const int64_t ks = (g.k + gridDim.y - 1) / gridDim.y;  // columns of this workgroup's slice
    const int64_t b0 = min((int64_t)blockIdx.y * ks, g.k), b1 = min(b0 + ks, g.k);
    const int64_t kc = (b1 - b0 + kGemvRowsWaves - 1) / kGemvRowsWaves;
    const int64_t c0 = min(b0 + (int64_t)w * kc, b1), c1 = min(c0 + kc, b1);
    d2 acc[4];
#pragma unroll
    for (int u = 0; u < 4; u++) acc[u] = (d2){0.0, 0.0};
    int64_t c = c0;
    for (; c + 4 <= c1; c += 4) {
        d2 v[4];
        double x[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            v[u] = *reinterpret_cast<const d2 *>(row + g.mcofs[c + u]);
            x[u] = g.X[op_addr<kVK>(g.xv, 0, c + u)];
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            acc[u].x = fma(v[u].x, x[u], acc[u].x);
            acc[u].y = fma(v[u].y, x[u], acc[u].y);
        }
    }
    for (int u = 0; c < c1; c++, u++) {
        const d2 v = *reinterpret_cast<const d2 *>(row + g.mcofs[c]);
        const double x = g.X[op_addr<kVK>(g.xv, 0, c)];
        acc[u].x = fma(v.x, x, acc[u].x);
        acc[u].y = fma(v.y, x, acc[u].y);
    }
    red[w][lane] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
    __syncthreads();
    if (w != 0 || pr >= npairs) return;
    d2 sum = red[0][lane];
#pragma unroll
    for (int q = 1; q < kGemvRowsWaves; q++) sum += red[q][lane];
    if (gridDim.y > 1) {
        *reinterpret_cast<d2 *>(ws + (int64_t)blockIdx.y * g.rows + 2 * pr) = sum;
        return;
    }
    gemv_store(g, 2 * pr, g.alpha * sum.x);
    gemv_store(g, 2 * pr + 1, g.alpha * sum.y);
}

__global__ __launch_bounds__(256) void gemv_rows_reduce(GemvArgs g, const double *ws, uint32_t nslice)
{
    const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (r >= g.rows) return;
    gemv_store(g, r, g.alpha * sum_in_order(ws + r, nslice, g.rows));
}

// Thin products (ThinArgs): C (rows x nt) = alpha * T S^T with T the long
// operand (rows x k, k short) and S the thin one (nt x k; nt <= 48, or up
// to 192 when k <= 48).  Every element of T is used once, so the product
// is bound by streaming T from HBM, by the FP64 MFMA rate (about as fast at
// nt = 48) or, at wide nt and short k, by writing C; tiles of 64 x 64
// re-read S per tile and keep too few loads in flight (3 TB/s).
// Here S lives in LDS for the whole launch, pre-arranged as the MFMA
// fragments of every 8-wide K chunk (two per chunk, t = 0, 1, one read of
// 512 contiguous bytes each) and 16-wide block of S rows, and each wave
// streams units of 32 rows of T through registers: a unit's K is read in
// super chunks of kThinSC chunks (two 16-byte loads per lane per 8-wide
// chunk), the next super chunk (of this unit or the wave's next) loading
// while this one runs its MFMAs.  With nt > 48 (k <= 48: one super chunk)
// the unit's registers serve ng groups of 48 S rows in turn.
//   KP (k pairs adjacent, kDK / kVK): lane (i = l%16, q = l/16) loads
//     T[r][k0 + 2q], T[r][k0 + 2q + 1] for r = row0 + i (row block 0) and
//     r = row0 + 16 + i (block 1); component x pairs with fragment t = 0
//     (k = k0 + 2q), y with t = 1.
//   !KP (row pairs adjacent, kDMN / kVMN): lane loads T[row0 + 2i][k],
//     T[row0 + 2i + 1][k] for k = k0 + q (t = 0) and k0 + 4 + q (t = 1);
//     x feeds row block 0 (even rows), y block 1 (odd rows).
// The register fragment is the MFMA's A operand (T rows down the result,
// S rows across: lanes of a store run along S) or, TC, its B operand (the
// result transposed: lanes run along T), chosen so a store's 16 lanes
// write consecutive addresses of C: TC when C(r, j) is C's column r (the
// product of a thin A, written transposed).
// Both sum every C element over k in a fixed order, independent of timing.
// No load's result is used in the item that issues it (the compiler's
// in-order load counter would otherwise make every MFMA of that item wait
// for the prefetch as well): the row offsets of a unit are loaded one item
// ahead into one of two register sets, the T side's C offsets of the unit
// being computed are loaded at the start of each item, the S side's sit in
// LDS, and every load is unconditional (past the wave's last item and past
// K they repeat valid addresses).
// Registers: two super chunks (96), 2 x NBB accumulators and the offsets;
// NBB = 4 would spill at two waves per SIMD, so a group is 48 wide.
constexpr int kThinSC = 6;
struct ThinArgs {
    int64_t rows, nt, k;
    int32_t ng;  // groups of 16 * NBB rows of S
    double alpha;
    const double *T;
    OpArgs t;
    int32_t tdense;  // T dense (ld) or a view without block table
    const double *S;
    OpArgs s;
    int32_t smode;   // kDK, kDMN or a view mode
    double *C;
    OpArgs c;
    int32_t cview, ctr;  // ctr: element (r, j) of the product is C(j, r); views have no block table
    int32_t cpair;       // ctr: C(j, r), C(j, r + 1) adjacent and 16-byte aligned for even r
    int32_t overwrite;
};

__device__ inline double thin_s(const ThinArgs &g, int64_t j, int64_t kk)
{
    if (g.smode == kDK) return g.S[j * g.s.ld + kk];
    if (g.smode == kDMN) return g.S[kk * g.s.ld + j];
    return g.S[op_addr<kVK>(g.s, j, kk)];
}

// TD: T dense; CV: C a view; TC: transposed C (ctr), the transposed MFMA
// form.  Compile-time, so no load sits in a branch whose other side writes
// the same register, which would force a full wait.
template <bool KP, int NBB, bool TD, bool CV, bool TC>
__global__ __launch_bounds__(256, 2) void thin_kernel(ThinArgs g)
{
    extern __shared__ double smem[];
    const int64_t K = g.k;
    const int NBT = g.ng * NBB;  // 16-row blocks of S
    double *bf = smem;           // [K / 8][t][NBT][64 lanes]
    int64_t *cp = reinterpret_cast<int64_t *>(smem + K * NBT * 16);  // column part of T per k
    int64_t *cthin = cp + K;                                         // C offset per S row
    const int tid = threadIdx.x, lane = tid & 63, i16 = lane & 15, q = lane >> 4;

    for (int64_t e = tid; e < K * NBT * 16; e += 256) {
        const int l = (int)(e & 63);
        const int64_t f = e >> 6;
        const int cb = (int)(f % NBT), t = (int)((f / NBT) & 1);
        const int64_t c = f / NBT / 2;
        const int64_t j = 16 * cb + (l & 15), kk = KP ? 8 * c + 2 * (l >> 4) + t : 8 * c + 4 * t + (l >> 4);
        bf[e] = j < g.nt ? thin_s(g, j, kk) : 0.0;
    }
    for (int64_t c = tid; c < K; c += 256) {
        if constexpr (!TD) cp[c] = g.t.cofs[c];
        else cp[c] = KP ? c : c * g.t.ld;
    }
    for (int j = tid; j < 16 * NBT; j += 256) {
        const int64_t jj = min((int64_t)j, g.nt - 1);
        if constexpr (CV) cthin[j] = TC ? g.c.rofs[jj] : g.c.cofs[jj];
        else cthin[j] = TC ? jj * g.c.ld : jj;
    }
    __syncthreads();

    const int64_t U = (g.rows + 31) / 32, NW = (int64_t)gridDim.x * 4;
    int64_t cu = (int64_t)blockIdx.x * 4 + (tid >> 6);
    if (cu >= U) return;
    const int nsc = (int)((K + 8 * kThinSC - 1) / (8 * kThinSC));

    // Row parts of T for unit u in this lane (rows past the end load the
    // last row or row pair: in range, never stored).
    auto row_part = [&](int64_t r) -> int64_t {
        if constexpr (!TD) return g.t.rofs[r];
        else return KP ? r * g.t.ld : r;
    };
    auto rows_of = [&](int64_t u, int64_t (&p)[2]) __attribute__((always_inline)) {
        if constexpr (KP) {
            p[0] = row_part(min(u * 32 + i16, g.rows - 1));
            p[1] = row_part(min(u * 32 + 16 + i16, g.rows - 1));
        } else {
            p[0] = row_part(min(u * 32 + 2 * i16, g.rows - 2));
            p[1] = 0;
        }
    };
    // MFMA result: lane l, element r holds result row q + 4r, column i16.
    // The T row of element r of row block b (TC: the same for every r) and
    // the S row of element r of 16-row block jb of S.
    auto t_row = [&](int64_t u, int b, int r) -> int64_t {
        const int loc = TC ? i16 : q + 4 * r;
        return KP ? u * 32 + 16 * b + loc : u * 32 + 2 * loc + b;
    };
    auto s_row = [&](int jb, int r) -> int { return 16 * jb + (TC ? q + 4 * r : i16); };
    constexpr int NO = TC ? 1 : 4;  // distinct T rows per row block and lane
    // Rows past the end are clamped into range; with row pairs the even row
    // clamps to rows - 2 (rows is even), so a clamped pair stays a whole,
    // aligned pair.
    auto c_offsets = [&](int64_t u, int64_t (&o)[2][NO]) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int r = 0; r < NO; r++) {
                const int64_t row = KP ? min(t_row(u, b, r), g.rows - 1) : min(t_row(u, 0, r), g.rows - 2) + b;
                if constexpr (CV) o[b][r] = (TC ? g.c.cofs : g.c.rofs)[row];
                else o[b][r] = TC ? row : row * g.c.ld;
            }
    };
    auto load = [&](d2 (&a)[2 * kThinSC], const int64_t (&p)[2], int sc) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < kThinSC; c++) {
            const int64_t k0 = min((int64_t)(8 * kThinSC * sc + 8 * c), K - 8);
            if constexpr (KP) {
                const int64_t co = cp[k0 + 2 * q];
                a[2 * c] = *reinterpret_cast<const d2 *>(g.T + p[0] + co);
                a[2 * c + 1] = *reinterpret_cast<const d2 *>(g.T + p[1] + co);
            } else {
                a[2 * c] = *reinterpret_cast<const d2 *>(g.T + p[0] + cp[k0 + q]);
                a[2 * c + 1] = *reinterpret_cast<const d2 *>(g.T + p[0] + cp[k0 + 4 + q]);
            }
        }
    };
    d4 acc[2][NBB];
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
        for (int j = 0; j < NBB; j++) acc[b][j] = (d4){0.0, 0.0, 0.0, 0.0};
    auto mma = [&](double tv, double sv, d4 c) -> d4 {
        if constexpr (TC) return __builtin_amdgcn_mfma_f64_16x16x4f64(sv, tv, c, 0, 0, 0);
        else return __builtin_amdgcn_mfma_f64_16x16x4f64(tv, sv, c, 0, 0, 0);
    };
    auto compute = [&](const d2 (&a)[2 * kThinSC], int sc, int grp) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < kThinSC; c++) {
            const int64_t kc = kThinSC * sc + c;
            if (8 * kc >= K) break;
#pragma unroll
            for (int j = 0; j < NBB; j++) {
                const int jb = grp * NBB + j;
                const double b0 = bf[((kc * 2) * NBT + jb) * 64 + lane];
                const double b1 = bf[((kc * 2 + 1) * NBT + jb) * 64 + lane];
                if constexpr (KP) {
                    acc[0][j] = mma(a[2 * c].x, b0, acc[0][j]);
                    acc[1][j] = mma(a[2 * c + 1].x, b0, acc[1][j]);
                    acc[0][j] = mma(a[2 * c].y, b1, acc[0][j]);
                    acc[1][j] = mma(a[2 * c + 1].y, b1, acc[1][j]);
                } else {
                    acc[0][j] = mma(a[2 * c].x, b0, acc[0][j]);
                    acc[1][j] = mma(a[2 * c].y, b0, acc[1][j]);
                    acc[0][j] = mma(a[2 * c + 1].x, b1, acc[0][j]);
                    acc[1][j] = mma(a[2 * c + 1].y, b1, acc[1][j]);
                }
            }
        }
    };
    // Accumulating into C reads a row block's old values with one batch of
    // loads (clamped addresses, all in range) and one wait.  Row pairs in
    // the transposed form: a lane's two row blocks hold T rows 2i and 2i + 1,
    // adjacent in C, so with cpair they go out as one 16-byte store (two
    // 8-byte stores a row apart left half-written lines for L2 to write
    // back, 1.5x the bytes).
    auto store = [&](int64_t u, const int64_t (&o)[2][NO], int grp) __attribute__((always_inline)) {
        if constexpr (!KP && TC) {
            if (g.cpair) {
                const bool rin = t_row(u, 0, 0) < g.rows;  // rows are even: the pair is whole
                d2 old2[NBB][4];
                if (!g.overwrite) {
#pragma unroll
                    for (int j = 0; j < NBB; j++)
#pragma unroll
                        for (int r = 0; r < 4; r++)
                            old2[j][r] = *reinterpret_cast<const d2 *>(
                                g.C + o[0][0] + cthin[s_row(grp * NBB + j, r)]);
                }
#pragma unroll
                for (int j = 0; j < NBB; j++) {
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int sr = s_row(grp * NBB + j, r);
                        if (!rin || sr >= g.nt) continue;
                        d2 v = {g.alpha * acc[0][j][r], g.alpha * acc[1][j][r]};
                        if (!g.overwrite) v = old2[j][r] + v;
                        *reinterpret_cast<d2 *>(g.C + o[0][0] + cthin[sr]) = v;
                    }
                    acc[0][j] = (d4){0.0, 0.0, 0.0, 0.0};
                    acc[1][j] = (d4){0.0, 0.0, 0.0, 0.0};
                }
                return;
            }
        }
#pragma unroll
        for (int b = 0; b < 2; b++) {
            double old[NBB][4];
            if (!g.overwrite) {
#pragma unroll
                for (int j = 0; j < NBB; j++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        old[j][r] = g.C[o[b][TC ? 0 : r] + cthin[s_row(grp * NBB + j, r)]];
            }
#pragma unroll
            for (int j = 0; j < NBB; j++) {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int sr = s_row(grp * NBB + j, r);
                    if (t_row(u, b, r) >= g.rows || sr >= g.nt) continue;
                    const double v = g.alpha * acc[b][j][r];
                    g.C[o[b][TC ? 0 : r] + cthin[sr]] = g.overwrite ? v : old[j][r] + v;
                }
                acc[b][j] = (d4){0.0, 0.0, 0.0, 0.0};
            }
        }
    };

    // The wave's items (unit, super chunk) in order; item n + 1 loads while
    // item n computes.  p: row parts of the unit being loaded; qa / qb: those
    // of the unit after it, loaded by alternate items and used one item
    // later.  Unit indices past the end are clamped, so every item issues
    // the same loads.
    int64_t p[2], qa[2], qb[2], co[2][NO];
    rows_of(cu, p);
    rows_of(min(cu + NW, U - 1), qb);
    d2 ra[2 * kThinSC], rb[2 * kThinSC];
    load(ra, p, 0);
    int cs = 0;
    auto next = [&](d2 (&a)[2 * kThinSC], int64_t (&qload)[2], const int64_t (&quse)[2], int64_t &lu,
                    int &ls) __attribute__((always_inline)) {
        c_offsets(cu, co);
        lu = cu;
        ls = cs + 1;
        if (ls == nsc) {
            ls = 0;
            lu += NW;
        }
        const bool nu = ls == 0;
        p[0] = nu ? quse[0] : p[0];
        p[1] = nu ? quse[1] : p[1];
        rows_of(min(lu + NW, U - 1), qload);
        load(a, p, ls);
    };
    // One item: every group of S rows (several only with one super chunk).
    auto work = [&](const d2 (&a)[2 * kThinSC]) __attribute__((always_inline)) {
        for (int grp = 0; grp < g.ng; grp++) {
            compute(a, cs, grp);
            if (cs == nsc - 1) store(cu, co, grp);
        }
    };
    while (true) {
        int64_t lu;
        int ls;
        next(rb, qa, qb, lu, ls);
        work(ra);
        if (lu >= U) break;
        cu = lu;
        cs = ls;

        next(ra, qb, qa, lu, ls);
        work(rb);
        if (lu >= U) break;
        cu = lu;
        cs = ls;
    }
}

}  // namespace

int gemv_f64_launch(const GemvArgs &g, hipStream_t s)
{
    DTCF_REQUIRE(g.k > 0 && g.k % 2 == 0 && g.k <= kGemvMaxK, "gemv: k must be even and <= 20480");
    if (g.rows <= 0) return DTCF_OK;
    static std::once_flag once;
    static hipError_t attr_err = hipSuccess;
    std::call_once(once, [&] {
        attr_err = hipFuncSetAttribute(reinterpret_cast<const void *>(gemv_kernel),
                                       hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)(kGemvMaxK * sizeof(double)));
    });
    DTCF_HIP(attr_err);
    const unsigned grid = (unsigned)std::min<int64_t>((g.rows + 3) / 4, 2048);
    hipLaunchKernelGGL(gemv_kernel, dim3(grid), dim3(256), (size_t)g.k * sizeof(double), s, g);
    DTCF_HIP(hipGetLastError());
    return DTCF_OK;
}

// 16-row blocks of S a thin product keeps in LDS (0: not a thin shape).
static int64_t thin_blocks(int64_t w, int64_t k)
{
    if (w <= kThinMaxWidth) return (w + 15) / 16;
    if (w <= kThinMaxWide && k <= kThinWideK) return 3 * ((w + 47) / 48);
    return 0;
}

bool thin_shape(int64_t m, int64_t n, int64_t k, int64_t min_rows)
{
    const int64_t w = std::min(m, n), rows = std::max(m, n);
    const int64_t nbt = thin_blocks(w, k);
    if (nbt == 0 || rows < min_rows || k <= 0 || k % 8 != 0) return false;
    return (k * 16 * nbt + k + 16 * nbt) * (int64_t)sizeof(double) <= kThinLdsBytes;
}

template <bool KP, int NBB, bool TD, bool CV, bool TC>
int thin_launch_t(const ThinArgs &t, hipStream_t s)
{
    auto kern = thin_kernel<KP, NBB, TD, CV, TC>;
    static std::once_flag once;
    static hipError_t attr_err = hipSuccess;
    std::call_once(once, [&] {
        attr_err = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)kThinLdsBytes);
    });
    DTCF_HIP(attr_err);
    int cus = 0;
    const int st = gemm_device_cus(&cus);
    if (st != DTCF_OK) return st;
    // Two resident workgroups per CU (LDS up to 80 KiB each), each wave
    // looping over 32-row units.
    const int64_t units = (t.rows + 31) / 32, nbt = (int64_t)t.ng * NBB;
    const unsigned grid = (unsigned)std::min<int64_t>((units + 3) / 4, (int64_t)cus * 2);
    const size_t lds = (size_t)(t.k * 16 * nbt + t.k + 16 * nbt) * sizeof(double);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(256), lds, s, t);
    DTCF_HIP(hipGetLastError());
    return DTCF_OK;
}

template <bool KP, bool TD, bool CV, bool TC>
int thin_dispatch_nbb(const ThinArgs &t, int nbb, hipStream_t s)
{
    if (nbb == 1) return thin_launch_t<KP, 1, TD, CV, TC>(t, s);
    if (nbb == 2) return thin_launch_t<KP, 2, TD, CV, TC>(t, s);
    return thin_launch_t<KP, 3, TD, CV, TC>(t, s);
}

template <bool KP, bool TD>
int thin_dispatch(const ThinArgs &t, int nbb, hipStream_t s)
{
    if (t.cview) {
        if (t.ctr) return thin_dispatch_nbb<KP, TD, true, true>(t, nbb, s);
        return thin_dispatch_nbb<KP, TD, true, false>(t, nbb, s);
    }
    if (t.ctr) return thin_dispatch_nbb<KP, TD, false, true>(t, nbb, s);
    return thin_dispatch_nbb<KP, TD, false, false>(t, nbb, s);
}

int thin_f64_launch(const GemmArgs &g, hipStream_t s)
{
    // The long operand: A when n is the thin side, else B (C written
    // transposed).
    const bool tall_a = g.m >= g.n;
    ThinArgs t{};
    t.rows = tall_a ? g.m : g.n;
    t.nt = tall_a ? g.n : g.m;
    t.k = g.k;
    if (!thin_shape(t.rows, t.nt, t.k, 1)) return kThinDecline;
    const OpArgs &to = tall_a ? g.a : g.b;
    const int tmode = tall_a ? g.amode : g.bmode;
    const bool kp = tmode == kDK || tmode == kVK;
    if (!to.vec2 || (tmode >= kVK && to.blk) || (!kp && t.rows % 2 != 0)) return kThinDecline;
    if (g.cview && g.c.blk) return kThinDecline;
    const int64_t nbt = thin_blocks(t.nt, t.k);
    const int nbb = (int)std::min<int64_t>(nbt, 3);
    t.ng = (int32_t)(nbt / nbb);
    t.alpha = g.alpha;
    t.T = tall_a ? g.A : g.B;
    t.t = to;
    t.tdense = tmode <= kDMN;
    t.S = tall_a ? g.B : g.A;
    t.s = tall_a ? g.b : g.a;
    t.smode = tall_a ? g.bmode : g.amode;
    t.C = g.C;
    t.c = g.c;
    t.cview = g.cview;
    t.ctr = tall_a ? 0 : 1;
    t.cpair = tall_a ? 0
                     : (g.cview ? g.c.vec2
                                : ((reinterpret_cast<uintptr_t>(g.C) & 15) == 0 && g.c.ld % 2 == 0));
    t.overwrite = g.overwrite;
    if (kp) {
        if (t.tdense) return thin_dispatch<true, true>(t, nbb, s);
        return thin_dispatch<true, false>(t, nbb, s);
    }
    if (t.tdense) return thin_dispatch<false, true>(t, nbb, s);
    return thin_dispatch<false, false>(t, nbb, s);
}

int gemv_rows_f64_launch(const GemvArgs &g, hipStream_t s)
{
    DTCF_REQUIRE(g.k > 0 && g.rows % 2 == 0, "gemv rows: k must be positive and the row count even");
    if (g.rows <= 0) return DTCF_OK;
    const int64_t blocks = (g.rows / 2 + 63) / 64;
    DTCF_REQUIRE(blocks < (1ll << 31), "gemv rows: too many rows");
    int cus = 0;
    int st = gemm_device_cus(&cus);
    if (st != DTCF_OK) return st;
    // Column slices over workgroups until the grid covers two workgroups
    // per CU, each slice keeping at least 64 columns per wave.
    int64_t nslice = 1;
    while (blocks * nslice < 2 * (int64_t)cus && g.k / (2 * nslice) >= 64 * kGemvRowsWaves) nslice *= 2;
    double *ws = nullptr;
    if (nslice > 1) {
        st = gemm_workspace(s, (size_t)nslice * g.rows * sizeof(double), &ws);
        if (st != DTCF_OK) return st;
    }
    hipLaunchKernelGGL(gemv_rows_kernel, dim3((unsigned)blocks, (unsigned)nslice), dim3(64 * kGemvRowsWaves), 0,
                       s, g, ws);
    DTCF_HIP(hipGetLastError());
    if (nslice > 1) {
        hipLaunchKernelGGL(gemv_rows_reduce, dim3((unsigned)((g.rows + 255) / 256)), dim3(256), 0, s, g,
                           (const double *)ws, (uint32_t)nslice);
        DTCF_HIP(hipGetLastError());
    }
    return DTCF_OK;
}

}  // namespace dtcf
