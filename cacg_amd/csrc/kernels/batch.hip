// Batched kernels: one launch advances a phase of the s-step iteration for
// every system in a work list (the batching / serving form).  gfx950, wave64.
//
// Systems of the batch differ in n, nnz, m (<= 32) and sm = s*m (<= 128), so
// the SpMM kernels map lanes to the elements (row, column) of a 64-row tile:
// lane e of the tile handles row e / k, column e % k, which keeps every lane
// busy for any k.  The dense products (Gram blocks, Q = S - Q beta,
// X += Q alpha) run on FP64 MFMA over 2048-row chunks: the Gram in one launch for
// every width, a chunk's output tiles split over waves; the updates with one
// launch per tile class (the system's sm and m rounded up to 16-column tiles,
// zero-padded), a chunk's rows split until the launch fills the chip.  A second
// kernel sums the Gram chunk partials in chunk order.  Every sum of a system runs
// in an order fixed by that system alone (its rows, tiles, chunks and class), so a
// system's results are the same bits whatever else shares the launch.
// 64 systems, FP32 basis: 252 -> 116 ms; the Gram of a full round 1110 -> about 300
// us, Q updates 830 -> 240, X updates 546 -> 118.
#include <type_traits>

#include "kcommon.hpp"

namespace {

constexpr int BT = CACG_BT;
constexpr int GR = CACG_GR;
constexpr int GS = 16;  // rows per LDS stage of the Gram
constexpr int MS = CACG_BATCH_MAX_SM, MM = CACG_BATCH_MAX_M;

__device__ __forceinline__ int tile_rows(int n, int tile)
{
    const int r = n - tile * BT;
    return r < BT ? r : BT;
}

// sum over row i of val[p] * x[col[p] * ldx + c] in CSR order, products and sums
// rounded separately (the reference's SpMM arithmetic); the gathers of 8
// nonzeros are issued before they are accumulated, for memory-level parallelism
template <typename TV, typename TX>
__device__ __forceinline__ TV row_dot(const int *__restrict__ rowptr, const int *__restrict__ col,
                                      const TV *__restrict__ val, const TX *__restrict__ x, long ldx,
                                      int c, long i)
{
    const int pb = rowptr[i], pe = rowptr[i + 1];
    TV acc = (TV)0;
    for (int p = pb; p < pe; p += 8) {
        int cc[8];
        TV vv[8];
        TX xv[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const bool in = p + u < pe;
            cc[u] = in ? col[p + u] : 0;
            vv[u] = in ? val[p + u] : (TV)0;
        }
#pragma unroll
        for (int u = 0; u < 8; u++)
            xv[u] = p + u < pe ? x[(long)cc[u] * ldx + c] : (TX)0;
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (p + u < pe)
                acc = add_rn(acc, mul_rn(vv[u], (TV)xv[u]));
    }
    return acc;
}

// Vector path of the tile SpMMs: the tile's row pointers and (col, val)
// pairs staged in LDS (when at most CAPB), each lane producing 4 adjacent
// columns of one row from 16-byte gathers of x, 4 nonzeros gathered ahead of
// their in-order accumulation.  Each output is the CSR-order sum of separately
// rounded products, the bits of row_dot.
constexpr int CAPB = 1024;

template <typename TV>
struct TileCsr {
    int rp[BT + 1];
    int col[CAPB];
    TV val[CAPB];
};

// stage rows r0 .. r0 + rows - 1; returns whether the pairs fit (else the
// caller uses row_dot); ends with a barrier
template <typename TV>
__device__ __forceinline__ bool stage_tile(TileCsr<TV> &tc, const int *__restrict__ rowptr,
                                           const int *__restrict__ col,
                                           const TV *__restrict__ val, long r0, int rows)
{
    for (int e = threadIdx.x; e <= rows; e += 256)
        tc.rp[e] = rowptr[r0 + e];
    __syncthreads();
    const int pb = tc.rp[0], tn = tc.rp[rows] - pb;
    const bool staged = tn <= CAPB;
    if (staged)
        for (int e = threadIdx.x; e < tn; e += 256) {
            tc.col[e] = col[pb + e];
            tc.val[e] = val[pb + e];
        }
    __syncthreads();
    return staged;
}

// 4 elements of x converted to TV: p[0..3] (FP32, one 16-byte load), or the
// FP64 pairs p[0..1] and p[off..off+1] (16-byte aligned)
template <typename TV, typename TX>
__device__ __forceinline__ void load4(const TX *p, TV *o, int off)
{
    if constexpr (sizeof(TX) == 4) {
        const float4 v = *reinterpret_cast<const float4 *>(p);
        o[0] = (TV)v.x;
        o[1] = (TV)v.y;
        o[2] = (TV)v.z;
        o[3] = (TV)v.w;
    } else {
        const double2 v0 = *reinterpret_cast<const double2 *>(p);
        const double2 v1 = *reinterpret_cast<const double2 *>(p + off);
        o[0] = (TV)v0.x;
        o[1] = (TV)v0.y;
        o[2] = (TV)v1.x;
        o[3] = (TV)v1.y;
    }
}

// Columns of a thread's 4 elements in an FP64 row block of width w (w % 4 == 0):
// the pairs c0, c0 + 1 and c0 + w / 2, c0 + w / 2 + 1 with c0 = 2 t for the
// t-th thread of the row, so each 16-byte access instruction of the threads of a
// row covers one contiguous half of it (FP32: 4 contiguous from 4 t).  Which
// thread computes an element changes no bit.
struct cols4 {
    int c0, off;
    __device__ __forceinline__ cols4(int t, int w, bool fp64)
        : c0(fp64 ? 2 * t : 4 * t), off(fp64 ? w / 2 : 2) {}
    __device__ __forceinline__ int operator()(int k) const { return k < 2 ? c0 + k : c0 + off + k - 2; }
};

// acc[0..3] = sums over row r of the staged tile of val * x[col * ldx + cs(0..3)]
template <typename TV, typename TX>
__device__ __forceinline__ void row_dot4(const TileCsr<TV> &tc, int r, const TX *__restrict__ x,
                                         long ldx, const cols4 &cs, TV *acc)
{
    const int pb = tc.rp[0], p0 = tc.rp[r] - pb, p1 = tc.rp[r + 1] - pb;
#pragma unroll
    for (int k = 0; k < 4; k++)
        acc[k] = (TV)0;
    for (int p = p0; p < p1; p += 4) {
        TV xv[4][4], vv[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const bool in = p + u < p1;
            vv[u] = in ? tc.val[p + u] : (TV)0;
            if (in)
                load4<TV, TX>(x + (long)tc.col[p + u] * ldx + cs.c0, xv[u], cs.off);
        }
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (p + u < p1)
#pragma unroll
                for (int k = 0; k < 4; k++)
                    acc[k] = add_rn(acc[k], mul_rn(vv[u], xv[u][k]));
    }
}

// basis step j for one tile (see cacg_kb_basis); TB = basis type
template <typename TB>
__global__ __launch_bounds__(256) void bbasis_kernel(const cacg_bsys *__restrict__ sys,
                                                     const int2 *__restrict__ items, int j)
{
    __shared__ TileCsr<TB> tc;
    const int2 it = items[blockIdx.x];
    const cacg_bsys &d = sys[it.x];
    const int n = d.n, m = d.m, sm = d.sm;
    const long r0 = (long)it.y * BT;
    const int rows = tile_rows(n, it.y);
    TB *S = reinterpret_cast<TB *>(d.S);
    const TB *val = sizeof(TB) == 4 ? reinterpret_cast<const TB *>(d.val32)
                                    : reinterpret_cast<const TB *>(d.val);
    const TB a1 = (TB)d.sa, b1 = (TB)d.sb, a2 = (TB)(2.0 * d.sa), b2 = (TB)(2.0 * d.sb);
    if (j == 0) {
        for (int e = threadIdx.x; e < rows * m; e += 256) {
            const int r = e / m, c = e - r * m;
            const long i = r0 + r;
            S[i * sm + c] = (TB)d.R[i * m + c];
        }
        return;
    }
    // the vector path: m a multiple of 4 (16-byte aligned rows and blocks)
    const bool vec = m % 4 == 0 && stage_tile<TB>(tc, d.rowptr, d.col, val, r0, rows);
    if (vec) {
        const int q = m / 4;
        constexpr bool f64 = sizeof(TB) == 8;
        for (int e = threadIdx.x; e < rows * q; e += 256) {
            const int r = e / q;
            const cols4 cs(e - r * q, m, f64);
            const long i = r0 + r;
            TB acc[4];
            if (j == 1) {
                // FP32 basis: the FP64 R read as 4 contiguous columns
                const cols4 cr = f64 ? cs : cols4(e - r * q, m, false);
                row_dot4<TB, double>(tc, r, d.R, m, cr, acc);
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const TB e1 = (TB)d.R[i * m + cr(k)];
                    S[i * sm + cr(k)] = e1;
                    S[i * sm + m + cr(k)] = add_rn(mul_rn(a1, acc[k]), mul_rn(b1, e1));
                }
            } else {
                const TB *xs = S + (long)(j - 1) * m;
                row_dot4<TB, TB>(tc, r, xs, sm, cs, acc);
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const TB e1 = xs[i * sm + cs(k)], e2 = S[i * sm + (long)(j - 2) * m + cs(k)];
                    S[i * sm + (long)j * m + cs(k)] =
                        sub_rn(add_rn(mul_rn(a2, acc[k]), mul_rn(b2, e1)), e2);
                }
            }
        }
        return;
    }
    for (int e = threadIdx.x; e < rows * m; e += 256) {
        const int r = e / m, c = e - r * m;
        const long i = r0 + r;
        if (j == 1) {
            const TB acc = row_dot<TB, double>(d.rowptr, d.col, val, d.R, m, c, i);
            const TB e1 = (TB)d.R[i * m + c];
            S[i * sm + c] = e1;
            S[i * sm + m + c] = add_rn(mul_rn(a1, acc), mul_rn(b1, e1));
        } else {
            const TB *xs = S + (long)(j - 1) * m;
            const TB acc = row_dot<TB, TB>(d.rowptr, d.col, val, xs, sm, c, i);
            const TB e1 = xs[i * sm + c], e2 = S[i * sm + (long)(j - 2) * m + c];
            S[i * sm + (long)j * m + c] = sub_rn(add_rn(mul_rn(a2, acc), mul_rn(b2, e1)), e2);
        }
    }
}

template <typename TB>
__global__ __launch_bounds__(256) void bq_from_s_kernel(const cacg_bsys *__restrict__ sys,
                                                        const int2 *__restrict__ items)
{
    const int2 it = items[blockIdx.x];
    const cacg_bsys &d = sys[it.x];
    const long base = (long)it.y * BT * d.sm;
    const int cnt = tile_rows(d.n, it.y) * d.sm;
    const TB *S = reinterpret_cast<const TB *>(d.S);
    for (int e = threadIdx.x; e < cnt; e += 256)
        d.Q[base + e] = (double)S[base + e];
}

__global__ __launch_bounds__(256) void baq_kernel(const cacg_bsys *__restrict__ sys,
                                                  const int2 *__restrict__ items)
{
    __shared__ TileCsr<double> tc;
    const int2 it = items[blockIdx.x];
    const cacg_bsys &d = sys[it.x];
    const int sm = d.sm;
    const long r0 = (long)it.y * BT;
    const int rows = tile_rows(d.n, it.y);
    if (sm % 4 == 0 && stage_tile<double>(tc, d.rowptr, d.col, d.val, r0, rows)) {
        const int q = sm / 4;
        for (int e = threadIdx.x; e < rows * q; e += 256) {
            const int r = e / q;
            const cols4 cs(e - r * q, sm, true);
            double acc[4];
            row_dot4<double, double>(tc, r, d.Q, sm, cs, acc);
            double *y = d.AQ + (r0 + r) * sm;
            *reinterpret_cast<double2 *>(y + cs.c0) = double2{acc[0], acc[1]};
            *reinterpret_cast<double2 *>(y + cs.c0 + cs.off) = double2{acc[2], acc[3]};
        }
        return;
    }
    for (int e = threadIdx.x; e < rows * sm; e += 256) {
        const int r = e / sm, c = e - r * sm;
        const long i = r0 + r;
        d.AQ[i * sm + c] = row_dot<double, double>(d.rowptr, d.col, d.val, d.Q, sm, c, i);
    }
}

// ---- Gram partials ------------------------------------------------------------------

// A round lists a few hundred chunks of 2048 rows at most, so the chip is filled
// by splitting a chunk's output tiles, not its rows, over waves: a wave owns one
// 16 x 16 tile (systems of up to BG_SMALL tiles) or 2 x 2 of them and feeds the
// MFMAs straight from global memory, lane l loading L and [R1 | R2] at row
// l / 16 of each step of 4 and its own columns, BgDepth steps ahead in registers.
// No LDS, no barrier; the rows that the 4 waves of a workgroup share come from
// L1, and grid.x is a multiple of 8, so a chunk's workgroups (grid.y) share an
// L2.  One launch serves every width.  Per tile the k-steps run in row order
// from zero (rows past the chunk are zeros), so a partial depends on the system
// alone.
constexpr int BG_SMALL = CACG_BGRAM_SMALL;

template <int MT, int NT>
struct BgDepth {   // steps in flight: about 2000 to 3000 cycles of MFMAs
    static constexpr int D = MT * NT == 1 ? 32 : MT * NT == 2 ? 20 : 12;
};

template <typename T1, int MT, int NT>
__device__ __forceinline__ void bgram_tiles(const double *const *pa0, long sa, const T1 *const *pb0,
                                            const long *sb, int rows, double *gp, int sm, int kr,
                                            int a0, int b0)
{
    constexpr int D = BgDepth<MT, NT>::D;
    const int lane = threadIdx.x & 63, lr = lane >> 4, lc = lane & 15;
    const double *pa[MT], *ea[MT];
    const T1 *pb[NT], *eb[NT];
    double va[D][MT];
    T1 vb[D][NT];
    dbl4 acc[MT][NT];
    // rows past the last: the last row is read again and zeros are multiplied
#pragma unroll
    for (int i = 0; i < MT; i++) {
        ea[i] = pa0[i] + (rows - 1L) * sa;
        pa[i] = pa0[i] + lr * sa;
#pragma unroll
        for (int j = 0; j < NT; j++)
            acc[i][j] = dbl4{0.0, 0.0, 0.0, 0.0};
    }
#pragma unroll
    for (int j = 0; j < NT; j++) {
        eb[j] = pb0[j] + (rows - 1L) * sb[j];
        pb[j] = pb0[j] + lr * sb[j];
    }
    int il = lr, im = lr;   // row of the next load, of the next step
    auto load = [&](auto edge, int d) {
        const bool in = !edge || il < rows;
#pragma unroll
        for (int i = 0; i < MT; i++) {
            va[d][i] = *(in ? pa[i] : ea[i]);
            pa[i] += 4 * sa;
        }
#pragma unroll
        for (int j = 0; j < NT; j++) {
            vb[d][j] = *(in ? pb[j] : eb[j]);
            pb[j] += 4 * sb[j];
        }
        il += 4;
    };
    auto step = [&](auto edge, int d) {
        const bool in = !edge || im < rows;
        double x[MT], y[NT];
#pragma unroll
        for (int i = 0; i < MT; i++)
            x[i] = in ? va[d][i] : 0.0;
#pragma unroll
        for (int j = 0; j < NT; j++)
            y[j] = in ? (double)vb[d][j] : 0.0;
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++)
                acc[i][j] = mfma16x16x4(x[i], y[j], acc[i][j]);
        im += 4;
    };
#pragma unroll
    for (int d = 0; d < D; d++) {
        load(std::true_type(), d);
        __builtin_amdgcn_sched_barrier(0);   // in this order: waits count loads
    }
    const int nk = (rows + 3) / 4, full = rows / 4;
    int k = 0;
    for (; k + 2 * D <= full; k += D) {
#pragma unroll
        for (int d = 0; d < D; d++) {
            step(std::false_type(), d);
            load(std::false_type(), d);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    for (; k < nk; k += D) {
#pragma unroll
        for (int d = 0; d < D; d++)
            if (k + d < nk) {
                step(std::true_type(), d);
                load(std::true_type(), d);
            }
    }
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int a = a0 + i * 16 + lr + 4 * r, b = b0 + j * 16 + lc;
                if (a < sm && b < kr)
                    gp[(long)a * kr + b] = acc[i][j][r];
            }
}

// WHICH 0: Q^T A S = AQ^T S, 1: Q^T [AQ | R]
template <typename TB, int WHICH>
__global__ __launch_bounds__(256) void bgram_kernel(const cacg_bsys *__restrict__ sys,
                                                    const int2 *__restrict__ items, int count)
{
    using T1 = typename std::conditional<WHICH == 1, double, TB>::type;
    if ((int)blockIdx.x >= count)
        return;
    const int2 it = items[blockIdx.x];
    const cacg_bsys &d = sys[it.x];
    const int m = d.m, sm = d.sm, kr = sm + (WHICH ? m : 0);
    const int tm = (sm + 15) / 16, tn = (kr + 15) / 16;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int ti, tj, mt = 1, nt = 1;   // the wave's first tile and how many
    if (tm * tn <= BG_SMALL) {
        const int tile = blockIdx.y * 4 + w;
        ti = tile / tn;
        tj = tile - ti * tn;
    } else {
        const int gn = (tn + 3) / 4, g = blockIdx.y / gn;
        ti = g * 4 + (w >> 1) * 2;
        tj = (blockIdx.y - g * gn) * 4 + (w & 1) * 2;
        mt = tm - ti >= 2 ? 2 : 1;
        nt = tn - tj >= 2 ? 2 : 1;
    }
    if (ti >= tm || tj >= tn)
        return;
    const int lc = threadIdx.x & 15;
    const long c0 = (long)it.y * GR;
    const int rows = d.n - c0 < GR ? (int)(d.n - c0) : GR;
    // columns past the last are clamped to it (their sums are not stored)
    const double *L = (WHICH ? d.Q : d.AQ) + c0 * sm;
    const T1 *R1 = (WHICH ? reinterpret_cast<const T1 *>(d.AQ) : reinterpret_cast<const T1 *>(d.S)) +
                   c0 * sm;
    const double *pa[2];
    const T1 *pb[2];
    long sb[2];
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int a = min((ti + u) * 16 + lc, sm - 1), b = min((tj + u) * 16 + lc, kr - 1);
        pa[u] = L + a;
        pb[u] = R1 + b;
        sb[u] = sm;
        if constexpr (WHICH == 1) {
            if (b >= sm) {
                pb[u] = d.R + c0 * m + (b - sm);
                sb[u] = m;
            }
        }
    }
    double *gp = d.gpart + (long)it.y * sm * kr;
    const int a0 = ti * 16, b0 = tj * 16;
    if (mt == 1 && nt == 1)
        bgram_tiles<T1, 1, 1>(pa, sm, pb, sb, rows, gp, sm, kr, a0, b0);
    else if (mt == 1)
        bgram_tiles<T1, 1, 2>(pa, sm, pb, sb, rows, gp, sm, kr, a0, b0);
    else if (nt == 1)
        bgram_tiles<T1, 2, 1>(pa, sm, pb, sb, rows, gp, sm, kr, a0, b0);
    else
        bgram_tiles<T1, 2, 2>(pa, sm, pb, sb, rows, gp, sm, kr, a0, b0);
}

// chunk-ordered sum of the partials, 256 result entries per workgroup
__global__ __launch_bounds__(256) void bgram_reduce_kernel(const cacg_bsys *__restrict__ sys,
                                                           const int2 *__restrict__ items,
                                                           int which)
{
    const int2 it = items[blockIdx.x];
    const cacg_bsys &d = sys[it.x];
    const int sm = d.sm, m = d.m;
    const int kr = sm + (which ? m : 0);
    const int e = it.y * 256 + threadIdx.x;
    if (e >= sm * kr)
        return;
    const long stride = (long)sm * kr;
    double acc = 0.0;
    for (int ch = 0; ch < d.nchunk; ch++)
        acc += d.gpart[ch * stride + e];
    const int a = e / kr, b = e - a * kr;
    if (which == 0)
        d.QtAS[(long)a * sm + b] = acc;
    else if (b < sm)
        d.QtAQ[(long)a * sm + b] = acc;
    else
        d.QtR[(long)a * m + (b - sm)] = acc;
}

// rows [c0, c1) of chunk `chunk` that part blockIdx.y of gridDim.y takes, whole
// multiples of `unit`; empty past the last.  Rows are independent in the
// updates: the split changes no bit, so it follows the launch.
struct part_rows {
    int c0, c1;
    __device__ __forceinline__ part_rows(int chunk, int n, int unit)
    {
        const int len = (GR / unit + (int)gridDim.y - 1) / (int)gridDim.y * unit;
        const int e = chunk * GR + GR < n ? chunk * GR + GR : n;
        c0 = chunk * GR + (int)blockIdx.y * len;
        c1 = c0 + len < e ? c0 + len : e;
    }
};

// Q = S - Q beta with FP64 MFMA for systems with 16 (SM / 16 - 1) < sm <= SM:
// a part of a 2048-row chunk per 512-lane workgroup, beta in LDS (zero-padded to
// SM x SM), each wave takes 16-row tiles of the chunk; the contraction index
// is permuted across the lane groups (group g supplies k = g SM/4 + t at step
// t), so each lane's A operand is SM/4 contiguous values of one row (16-byte
// loads when sm == SM, EXACT; guarded loads with zeros past sm otherwise),
// read before the tile is written (in place).  Per output the k order is
// fixed by the system alone.
template <typename TB, int SM, bool EXACT>
__global__ __launch_bounds__(512) void bqupdate_mfma_kernel(const cacg_bsys *__restrict__ sys,
                                                            const int2 *__restrict__ items)
{
    constexpr int KQ = SM / 4, NTL = SM / 16;
    extern __shared__ double bl[];  // SM x SM
    const int2 it = items[blockIdx.x];
    const cacg_bsys &d = sys[it.x];
    const int n = d.n, sm = EXACT ? SM : d.sm;
    for (int e = threadIdx.x; e < SM * SM; e += 512) {
        const int q = e / SM, c = e - q * SM;
        bl[e] = (q < sm && c < sm) ? d.beta[(long)q * sm + c] : 0.0;
    }
    __syncthreads();
    const TB *S = reinterpret_cast<const TB *>(d.S);
    double *Q = d.Q;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int lg = lane >> 4, lc = lane & 15;
    const part_rows pr(it.y, n, 128);
    const int c0 = pr.c0, c1 = pr.c1;
    for (int i0 = c0 + wave * 16; i0 < c1; i0 += 8 * 16) {
        const long arow = i0 + lc;
        double av[KQ];
        if (EXACT && arow < c1) {
            const double2 *src = reinterpret_cast<const double2 *>(Q + arow * SM + lg * KQ);
#pragma unroll
            for (int u = 0; u < KQ / 2; u++) {
                const double2 v = src[u];
                av[2 * u] = v.x;
                av[2 * u + 1] = v.y;
            }
        } else {
#pragma unroll
            for (int u = 0; u < KQ; u++) {
                const int k = lg * KQ + u;
                av[u] = (arow < c1 && k < sm) ? Q[arow * sm + k] : 0.0;
            }
        }
#pragma unroll 1
        for (int j = 0; j < NTL; j++) {
            const int c = j * 16 + lc;
            double sv[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const long i = i0 + lg + 4 * r;
                sv[r] = (i < c1 && c < sm) ? (double)S[i * sm + c] : 0.0;
            }
            dbl4 acc = {0.0, 0.0, 0.0, 0.0};
            const double *bcol = bl + (lg * KQ) * SM + c;
#pragma unroll
            for (int t = 0; t < KQ; t++)
                acc = mfma16x16x4(av[t], bcol[t * SM], acc);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const long i = i0 + lg + 4 * r;
                if (i < c1 && c < sm)
                    Q[i * sm + c] = sv[r] - acc[r];
            }
        }
    }
}

// X += Q alpha with FP64 MFMA for systems with 16 (SM / 16 - 1) < sm <= SM:
// a part of a 2048-row chunk per 256-lane workgroup, alpha (sm x m, m <= 16 NTM) in
// registers in the K-permuted order of the A operand (zeros past sm), 16-row
// tiles per wave; 16-byte Q loads when sm == SM (EXACT).
template <int SM, int NTM, bool EXACT>
__global__ __launch_bounds__(256) void bxupdate_mfma_kernel(const cacg_bsys *__restrict__ sys,
                                                            const int2 *__restrict__ items)
{
    constexpr int KQ = SM / 4;
    const int2 it = items[blockIdx.x];
    const cacg_bsys &d = sys[it.x];
    const int n = d.n, m = d.m, sm = EXACT ? SM : d.sm;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int lg = lane >> 4, lc = lane & 15;
    double alf[NTM][KQ];
#pragma unroll
    for (int j = 0; j < NTM; j++) {
        const int c = j * 16 + lc;
#pragma unroll
        for (int t = 0; t < KQ; t++) {
            const int k = lg * KQ + t;
            alf[j][t] = (c < m && k < sm) ? d.alpha[(long)k * m + c] : 0.0;
        }
    }
    const part_rows pr(it.y, n, 64);
    const int c0 = pr.c0, c1 = pr.c1;
    for (int i0 = c0 + wave * 16; i0 < c1; i0 += 4 * 16) {
        const long arow = i0 + lc;
        double av[KQ];
        if (EXACT && arow < c1) {
            const double2 *src = reinterpret_cast<const double2 *>(d.Q + arow * SM + lg * KQ);
#pragma unroll
            for (int u = 0; u < KQ / 2; u++) {
                const double2 v = src[u];
                av[2 * u] = v.x;
                av[2 * u + 1] = v.y;
            }
        } else {
#pragma unroll
            for (int u = 0; u < KQ; u++) {
                const int k = lg * KQ + u;
                av[u] = (arow < c1 && k < sm) ? d.Q[arow * sm + k] : 0.0;
            }
        }
#pragma unroll
        for (int j = 0; j < NTM; j++) {
            dbl4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int t = 0; t < KQ; t++)
                acc = mfma16x16x4(av[t], alf[j][t], acc);
            const int c = j * 16 + lc;
            if (c < m) {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const long i = i0 + lg + 4 * r;
                    if (i < c1)
                        d.X[i * m + c] += acc[r];
                }
            }
        }
    }
}

// R = B - A X in the reference's SpMM arithmetic, plus the tile's column sums
// of R^2 (rows in order)
__global__ __launch_bounds__(256) void bresid_kernel(const cacg_bsys *__restrict__ sys,
                                                     const int2 *__restrict__ items)
{
    __shared__ double sq[BT * MM];
    const int2 it = items[blockIdx.x];
    const cacg_bsys &d = sys[it.x];
    const int m = d.m;
    const long r0 = (long)it.y * BT;
    const int rows = tile_rows(d.n, it.y);
    for (int e = threadIdx.x; e < rows * m; e += 256) {
        const int r = e / m, c = e - r * m;
        const long i = r0 + r;
        const double acc = row_dot<double, double>(d.rowptr, d.col, d.val, d.X, m, c, i);
        const double rv = sub_rn(d.B[i * m + c], acc);
        d.R[i * m + c] = rv;
        sq[e] = rv * rv;
    }
    __syncthreads();
    if ((int)threadIdx.x < m) {
        double s = 0.0;
        for (int r = 0; r < rows; r++)
            s += sq[r * m + threadIdx.x];
        d.npart[(long)it.y * m + threadIdx.x] = s;
    }
}

// norm2[c] = sum over the system's tiles, in tile order
__global__ __launch_bounds__(64) void bnorm_kernel(const cacg_bsys *__restrict__ sys,
                                                   const int2 *__restrict__ items)
{
    const cacg_bsys &d = sys[items[blockIdx.x].x];
    const int c = threadIdx.x;
    if (c >= d.m)
        return;
    // tile order, as before; the loads of 16 tiles go out before their adds
    // (one dependent load per tile made a 1024-tile system take ~170 us)
    double s = 0.0;
    int t = 0;
    for (; t + 16 <= d.ntile; t += 16) {
        double v[16];
#pragma unroll
        for (int u = 0; u < 16; u++)
            v[u] = d.npart[(long)(t + u) * d.m + c];
#pragma unroll
        for (int u = 0; u < 16; u++)
            s += v[u];
    }
    for (; t < d.ntile; t++)
        s += d.npart[(long)t * d.m + c];
    d.norm2[c] = s;
}

}  // namespace

extern "C" int cacg_kb_basis(const cacg_bsys *d_sys, const int2 *d_tiles, int count, int j, int f32,
                             hipStream_t st)
{
    if (count <= 0)
        return 0;
    if (j < 0)
        return (int)hipErrorInvalidValue;
    if (f32)
        hipLaunchKernelGGL(bbasis_kernel<float>, dim3(count), dim3(256), 0, st, d_sys, d_tiles, j);
    else
        hipLaunchKernelGGL(bbasis_kernel<double>, dim3(count), dim3(256), 0, st, d_sys, d_tiles, j);
    CACG_LAUNCH_CHECK();
    return 0;
}

extern "C" int cacg_kb_q_from_s(const cacg_bsys *d_sys, const int2 *d_tiles, int count, int f32,
                                hipStream_t st)
{
    if (count <= 0)
        return 0;
    if (f32)
        hipLaunchKernelGGL(bq_from_s_kernel<float>, dim3(count), dim3(256), 0, st, d_sys, d_tiles);
    else
        hipLaunchKernelGGL(bq_from_s_kernel<double>, dim3(count), dim3(256), 0, st, d_sys, d_tiles);
    CACG_LAUNCH_CHECK();
    return 0;
}

extern "C" int cacg_kb_aq(const cacg_bsys *d_sys, const int2 *d_tiles, int count, hipStream_t st)
{
    if (count <= 0)
        return 0;
    hipLaunchKernelGGL(baq_kernel, dim3(count), dim3(256), 0, st, d_sys, d_tiles);
    CACG_LAUNCH_CHECK();
    return 0;
}

extern "C" int cacg_bgram_groups(int sm, int kr)
{
    const int tm = (sm + 15) / 16, tn = (kr + 15) / 16;
    return tm * tn <= BG_SMALL ? (tm * tn + 3) / 4 : ((tm + 3) / 4) * ((tn + 3) / 4);
}

extern "C" int cacg_kb_gram(const cacg_bsys *d_sys, const int2 *d_chunks, int nchunks, int groups,
                            int which, int f32, hipStream_t st)
{
    if (nchunks <= 0)
        return 0;
    if ((which != 0 && which != 1) || groups < 1 || groups > 65535)
        return (int)hipErrorInvalidValue;
    const dim3 grid((nchunks + 7) / 8 * 8, groups);
    if (which == 1)
        hipLaunchKernelGGL((bgram_kernel<double, 1>), grid, dim3(256), 0, st, d_sys, d_chunks, nchunks);
    else if (f32)
        hipLaunchKernelGGL((bgram_kernel<float, 0>), grid, dim3(256), 0, st, d_sys, d_chunks, nchunks);
    else
        hipLaunchKernelGGL((bgram_kernel<double, 0>), grid, dim3(256), 0, st, d_sys, d_chunks, nchunks);
    CACG_LAUNCH_CHECK();
    return 0;
}

// the systems of one tile class: tm = ceil(sm / 16), tn = ceil(kr / 16)
extern "C" int cacg_kb_gram_class(const cacg_bsys *d_sys, const int2 *d_chunks, int nchunks,
                                  int which, int f32, int tm, int tn, hipStream_t st)
{
    if (nchunks <= 0)
        return 0;
    if ((which != 0 && which != 1) || tm < 1 || tm > 8 || tn < tm || tn > tm + (which ? 2 : 0))
        return (int)hipErrorInvalidValue;
    return cacg_kb_gram(d_sys, d_chunks, nchunks, cacg_bgram_groups(16 * tm, 16 * tn), which, f32, st);
}

extern "C" int cacg_kb_gram_reduce(const cacg_bsys *d_sys, const int2 *d_blocks, int nblocks,
                                   int which, hipStream_t st)
{
    if (nblocks <= 0)
        return 0;
    hipLaunchKernelGGL(bgram_reduce_kernel, dim3(nblocks), dim3(256), 0, st, d_sys, d_blocks,
                       which);
    CACG_LAUNCH_CHECK();
    return 0;
}

// parts per chunk that bring `count` chunks to at most about `want` workgroups
static int chunk_parts(int count, int want, int most)
{
    const int p = want / count;
    return p < 1 ? 1 : p > most ? most : p;
}

extern "C" int cacg_kb_qupdate_class(const cacg_bsys *d_sys, const int2 *d_chunks, int count,
                                     int smp, int exact, int f32, hipStream_t st)
{
    if (count <= 0)
        return 0;
    const size_t shm = (size_t)smp * smp * sizeof(double);
    // parts: one workgroup per CU where beta takes its LDS, more where it does not
    const int parts = chunk_parts(count, shm > 81920 ? 256 : 512, 16);
#define CACG_QLAUNCH(TBV, SMV, EX)                                                                \
    do {                                                                                          \
        cacg_allow_lds(bqupdate_mfma_kernel<TBV, SMV, EX>, shm);                                  \
        hipLaunchKernelGGL((bqupdate_mfma_kernel<TBV, SMV, EX>), dim3(count, parts), dim3(512), shm, st, \
                           d_sys, d_chunks);                                                      \
    } while (0)
#define CACG_QCLASS(SMV)                                                                          \
    case SMV:                                                                                     \
        if (f32) {                                                                                \
            if (exact)                                                                            \
                CACG_QLAUNCH(float, SMV, true);                                                   \
            else                                                                                  \
                CACG_QLAUNCH(float, SMV, false);                                                  \
        } else {                                                                                  \
            if (exact)                                                                            \
                CACG_QLAUNCH(double, SMV, true);                                                  \
            else                                                                                  \
                CACG_QLAUNCH(double, SMV, false);                                                 \
        }                                                                                         \
        break;
    switch (smp) {
        CACG_QCLASS(16)
        CACG_QCLASS(32)
        CACG_QCLASS(48)
        CACG_QCLASS(64)
        CACG_QCLASS(80)
        CACG_QCLASS(96)
        CACG_QCLASS(112)
        CACG_QCLASS(128)
    default:
        return (int)hipErrorInvalidValue;
    }
#undef CACG_QCLASS
#undef CACG_QLAUNCH
    CACG_LAUNCH_CHECK();
    return 0;
}

extern "C" int cacg_kb_xupdate_class(const cacg_bsys *d_sys, const int2 *d_chunks, int count,
                                     int smp, int exact, int m, hipStream_t st)
{
    if (count <= 0)
        return 0;
    if (m < 1 || m > 32)
        return (int)hipErrorInvalidValue;
    const int parts = chunk_parts(count, 1024, 32);
#define CACG_XLAUNCH(SMV, NT, EX)                                                                 \
    hipLaunchKernelGGL((bxupdate_mfma_kernel<SMV, NT, EX>), dim3(count, parts), dim3(256), 0, st, d_sys, \
                       d_chunks)
#define CACG_XCLASS(SMV)                                                                          \
    case SMV:                                                                                     \
        if (m <= 16) {                                                                            \
            if (exact)                                                                            \
                CACG_XLAUNCH(SMV, 1, true);                                                       \
            else                                                                                  \
                CACG_XLAUNCH(SMV, 1, false);                                                      \
        } else {                                                                                  \
            if (exact)                                                                            \
                CACG_XLAUNCH(SMV, 2, true);                                                       \
            else                                                                                  \
                CACG_XLAUNCH(SMV, 2, false);                                                      \
        }                                                                                         \
        break;
    switch (smp) {
        CACG_XCLASS(16)
        CACG_XCLASS(32)
        CACG_XCLASS(48)
        CACG_XCLASS(64)
        CACG_XCLASS(80)
        CACG_XCLASS(96)
        CACG_XCLASS(112)
        CACG_XCLASS(128)
    default:
        return (int)hipErrorInvalidValue;
    }
#undef CACG_XCLASS
#undef CACG_XLAUNCH
    CACG_LAUNCH_CHECK();
    return 0;
}

extern "C" int cacg_kb_resid(const cacg_bsys *d_sys, const int2 *d_tiles, int count,
                             const int2 *d_sysitems, int nsys, hipStream_t st)
{
    if (count > 0) {
        hipLaunchKernelGGL(bresid_kernel, dim3(count), dim3(256), 0, st, d_sys, d_tiles);
        CACG_LAUNCH_CHECK();
    }
    if (nsys > 0) {
        hipLaunchKernelGGL(bnorm_kernel, dim3(nsys), dim3(64), 0, st, d_sys, d_sysitems);
        CACG_LAUNCH_CHECK();
    }
    return 0;
}
