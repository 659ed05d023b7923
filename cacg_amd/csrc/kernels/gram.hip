// Gram blocks G = L^T [R1 | R2] over tall-skinny row-major blocks
// (Q^T A S, Q^T A Q, Q^T R of src/BLAS3.c:699-758).  gfx950, wave64.
//
// Reference order: one lane per entry G[a][b], one sequential chain over all
// rows in row order, product and sum rounded separately: the reference's
// summation at one rank, bit for bit.  The chain bounds its time at n
// dependent steps whatever the number of entries.
//
// Fast order: split-K.  Workgroup x owns a contiguous chunk of rows and forms its
// partial of G with FP64 MFMA v_mfma_f64_16x16x4f64 (contraction index = row), kl_pad x
// kr_pad, its sums in row order; a second kernel sums the partials in chunk order, so
// the result is deterministic and independent of scheduling.  Three kernels share the
// shapes out (gram_fast):
//   gram_direct_kernel  up to 32 columns against 64 and not many rows: operands from
//                       memory straight to the matrix cores;
//   gram_lds_kernel     128 columns against 128 or 144: stages of 16 rows through LDS;
//   gram_tile_kernel    every other shape, through LDS.
// Either LDS kernel holds two stages in LDS and two more in registers.
#include <type_traits>

#include "gram_plan.hpp"
#include "kcommon.hpp"

namespace {

// One workgroup per NJ x 16 block of G; every entry's sum is one chain in row
// order (the reference's summation, bit for bit), so the kernel takes n steps
// whatever the grid and what counts is the length of a step.  A wave issues an
// FP64 instruction about every 8.5 cycles, dependent or not, so the chain
// lanes (64 entries a wave) do nothing but add and the other waves form the
// products: lane l of a producer holds column b0 + l % 16 of RL adjacent rows,
// the columns of L lie RL x NJ to 16 lanes, and v_fmac_f64 takes L's value from
// its lane by DPP (row_newbcast; product + 0 rounds as the product does).  Two
// rows' products go to LDS with one 16-byte write, which a chain lane takes
// with one 16-byte read, a batch ahead of its sums.  Producer lanes load GREF_D
// stages ahead into registers; a stage ends with a barrier that waits for LDS
// alone, so loads stay in flight, and the chain lanes cross it with a batch in
// registers.  With one chain wave, wave 4 does nothing else than the barriers:
// it shares the chain's SIMD, and a producer there costs the chain 6%.
// 262,144 rows, 128 x 144: 3.77 -> 1.70 ms (6.5 ns a row), 128 x 128 3.4 -> 1.50
// ms; the chain alone takes 3.7 ns a row, the producers alone 5.3 (products
// through LDS and, with every CU at work, 13 TB/s out of the L2s).  Slower:
// chain waves of 16 or 32 lanes (2.99, 2.53 ms), 9 producers, loads 2 or 8
// stages ahead (the same).
constexpr int GREF_D = 4;

template <int NJ>
struct GrefShape {
    static constexpr int CW = NJ > 4 ? 2 : 1;                     // chain waves: 0 .. CW - 1
    static constexpr int PW = 6;                                  // producer waves
    static constexpr int RL = NJ > 5 ? 2 : NJ > 2 ? 4 : 8;        // rows per producer lane and stage
    static constexpr int ROWS = 4 * PW * RL;                      // rows a stage: 48, 96 or 192
    static constexpr int NB = RL == 8 ? 12 : 6, BP = ROWS / NB / 2;   // batches a stage, row pairs each
    static constexpr int BUF = ROWS * NJ * 8;                     // double2 per buffer
    static constexpr int JP = NJ > 4 ? 8 : NJ > 2 ? 4 : 2;        // lanes per row of L
    static constexpr int RA = 16 / JP, NA = RL / RA;              // rows per load of L, loads
};

struct GrefSrc {
    const double *L;
    long ldl;
    int kl;
    const double *R1;
    long ld1;
    int kr1;
    const double *R2;
    long ld2;
    int kr2;
};

// a of lanes L0 .. L0 + 3 (or L0 alone) of each 16, times b.  s_nop: a DPP read
// comes two wait states after the write of its register.
template <int L0>
__device__ __forceinline__ void bcast_mul4(double *p, double a, double b)
{
    p[0] = p[1] = p[2] = p[3] = 0.0;
#define CACG_BM(r, l) "v_fmac_f64_dpp %" #r ", %4, %5 row_newbcast:%" #l " row_mask:0xf bank_mask:0xf\n\t"
    asm("s_nop 1\n\t" CACG_BM(0, 6) CACG_BM(1, 7) CACG_BM(2, 8) CACG_BM(3, 9)
        : "+&v"(p[0]), "+&v"(p[1]), "+&v"(p[2]), "+&v"(p[3])
        : "v"(a), "v"(b), "n"(L0), "n"(L0 + 1), "n"(L0 + 2), "n"(L0 + 3));
#undef CACG_BM
}
template <int L0>
__device__ __forceinline__ double bcast_mul(double a, double b)
{
    double p = 0.0;
    asm("s_nop 1\n\tv_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
        : "+&v"(p)
        : "v"(a), "v"(b), "n"(L0));
    return p;
}
template <int L0, int NJ>
__device__ __forceinline__ void bcast_row(double *p, double a, double b)
{
    if constexpr (NJ >= 4) {
        bcast_mul4<L0>(p, a, b);
        if constexpr (NJ > 4)
            bcast_row<L0 + 4, NJ - 4>(p + 4, a, b);
    } else {
        p[0] = bcast_mul<L0>(a, b);
        if constexpr (NJ > 1)
            bcast_row<L0 + 1, NJ - 1>(p + 1, a, b);
    }
}

// the LDS accesses of every wave before it are done, loads from memory may be
// in flight
__device__ __forceinline__ void lds_barrier()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// products of row pair U / 2, U / 2 + 1, .. of a lane's RL rows
template <int NJ, int U = 0>
__device__ __forceinline__ void gref_products(double2 *out, const double *va, const double *vb)
{
    using SH = GrefShape<NJ>;
    double x[NJ], y[NJ];
    bcast_row<U % SH::RA * SH::JP, NJ>(x, va[U / SH::RA], vb[U]);
    bcast_row<(U + 1) % SH::RA * SH::JP, NJ>(y, va[(U + 1) / SH::RA], vb[U + 1]);
#pragma unroll
    for (int j = 0; j < NJ; j++)
        out[U / 2 * NJ * 16 + j * 16] = make_double2(x[j], y[j]);
    if constexpr (U + 2 < SH::RL)
        gref_products<NJ, U + 2>(out, va, vb);
}

template <int NJ>
__global__ __launch_bounds__(512) void gram_ref_kernel(int n, GrefSrc s, int nbb,
                                                       double *__restrict__ G1,
                                                       double *__restrict__ G2)
{
    using SH = GrefShape<NJ>;
    constexpr int CH = NJ * 16;   // chains
    extern __shared__ double2 gref_lds[];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    // an XCD's workgroups take consecutive blocks, so they share columns of L
    const int q8 = gridDim.x >> 3, r8 = gridDim.x & 7, xcd = blockIdx.x & 7;
    const int id = xcd * q8 + (xcd < r8 ? xcd : r8) + (blockIdx.x >> 3);
    const int a0 = id / nbb * NJ, b0 = id % nbb * 16;
    const int kr = s.kr1 + s.kr2;
    const int nst = (int)(((unsigned)n + SH::ROWS - 1) / SH::ROWS);
    if (w >= SH::CW) {
        // with one chain wave, wave 4 (which shares its SIMD) only keeps the barriers
        const int wp = SH::CW == 2 ? w - 2 : w < 4 ? w - 1 : w == 4 ? -1 : w - 2;
        if (wp < 0) {
            for (int st = 0; st <= nst; st++)
                lds_barrier();
            return;
        }
        const int c = lane & 15;
        // columns past the last are clamped to it (their sums are not stored)
        const int a = min(a0 + min(c % SH::JP, NJ - 1), s.kl - 1), b = min(b0 + c, kr - 1);
        const long la = s.ldl, lb = b < s.kr1 ? s.ld1 : s.ld2;
        const unsigned r0 = (wp * 4 + (lane >> 4)) * SH::RL;   // first of the lane's rows of a stage
        unsigned il = r0, ip = r0;                             // of the next load, the next products
        const unsigned ra = c / SH::JP;
        const double *pa = s.L + a, *pb = b < s.kr1 ? s.R1 + b : s.R2 + (b - s.kr1);
        const double *const ea = pa + (n - 1L) * la, *const eb = pb + (n - 1L) * lb;
        pa += (r0 + ra) * la;
        pb += r0 * lb;
        double va[GREF_D][SH::NA], vb[GREF_D][SH::RL];
        // EDGE: rows past the last may come; the last row is read again and zero
        // products formed, which change no sum (no chain is ever -0)
        auto load = [&](auto edge, int d) {
#pragma unroll
            for (int k = 0; k < SH::NA; k++) {
                const double *q = pa + k * SH::RA * la;
                va[d][k] = *(!edge || il + ra + k * SH::RA < (unsigned)n ? q : ea);
            }
#pragma unroll
            for (int u = 0; u < SH::RL; u++) {
                const double *q = pb + u * lb;
                vb[d][u] = *(!edge || il + u < (unsigned)n ? q : eb);
            }
            pa += SH::ROWS * la;
            pb += SH::ROWS * lb;
            il += SH::ROWS;
        };
        double2 *const out = gref_lds + (r0 >> 1) * CH + c;
        auto produce = [&](auto edge, int buf, int d) {
            if constexpr (edge) {
                double xa[SH::NA], xb[SH::RL];
#pragma unroll
                for (int k = 0; k < SH::NA; k++)
                    xa[k] = ip + ra + k * SH::RA < (unsigned)n ? va[d][k] : 0.0;
#pragma unroll
                for (int u = 0; u < SH::RL; u++)
                    xb[u] = ip + u < (unsigned)n ? vb[d][u] : 0.0;
                gref_products<NJ>(out + buf * SH::BUF, xa, xb);
            } else {
                gref_products<NJ>(out + buf * SH::BUF, va[d], vb[d]);
            }
            ip += SH::ROWS;
        };
        // stage st + 1 while stage st is summed; the last turn forms a stage that
        // nothing reads
        auto stage = [&](auto edge, int d) {
            produce(edge, (d + 1) & 1, (d + 1) % GREF_D);
            load(edge, (d + 1) % GREF_D);
            lds_barrier();
        };
#pragma unroll
        for (int d = 0; d < GREF_D; d++) {
            load(std::true_type(), d);
            __builtin_amdgcn_sched_barrier(0);   // in this order: waits count loads
        }
        produce(std::true_type(), 0, 0);
        load(std::true_type(), 0);
        lds_barrier();
        const int inner = n / SH::ROWS - 2 * GREF_D - 1;   // loads reach stage st + 2 D
        int st = 0;
        for (; st <= inner; st += GREF_D) {
#pragma unroll
            for (int d = 0; d < GREF_D; d++)
                stage(std::false_type(), d);
        }
        for (; st < nst; st += GREF_D) {
#pragma unroll
            for (int d = 0; d < GREF_D; d++)
                if (st + d < nst)
                    stage(std::true_type(), d);
        }
        return;
    }
    __builtin_amdgcn_s_setprio(3);
    const int ch = w * 64 + lane;
    if (ch >= CH)
        return;
    const double2 *const col = gref_lds + ch;
    const double2 *p = col;
    double2 x[SH::BP], y[SH::BP];
    double acc = 0.0;
    auto read = [&](double2 *v, int b) {
#pragma unroll
        for (int u = 0; u < SH::BP; u++)
            v[u] = p[(b * SH::BP + u) * CH];
        __builtin_amdgcn_sched_barrier(0);   // ahead of the sums, and no further
    };
    auto sum = [&](const double2 *v) {
#pragma unroll
        for (int u = 0; u < SH::BP; u++) {
            acc = add_rn(acc, v[u].x);
            acc = add_rn(acc, v[u].y);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    lds_barrier();
    read(x, 0);
    for (int st = 0; st < nst; st++) {
#pragma unroll
        for (int b = 1; b < SH::NB; b += 2) {
            read(y, b);
            sum(x);
            if (b + 1 == SH::NB) {
                lds_barrier();
                p = col + ((st + 1) & 1) * SH::BUF;
                read(x, 0);
            } else {
                read(x, b + 1);
            }
            sum(y);
        }
    }
    const int a = a0 + (ch >> 4), b = b0 + (ch & 15);
    if (a < s.kl) {
        if (b < s.kr1)
            G1[(long)a * s.kr1 + b] = acc;
        else if (b < kr)
            G2[(long)a * s.kr2 + (b - s.kr1)] = acc;
    }
}

// ---- fast: split-K FP64 MFMA ------------------------------------------------

// the shapes taken with a block-major R1: from four groups of tiles on (49 columns of
// L, or fewer against more than 144), at most 320 columns together.  The kernels would
// read others; a narrower or wider basis stored block-major has not been measured.
bool blk_shape(const GramPlan &p, int kl, int kr1) { return p.KS == 1 && kl + kr1 <= 320; }

// L (Q, AQ) and R2 (the residual R) are FP64, R1 FP64 or FP32 (AQ; the basis S, FP32 in
// the precision form).  Loaded values are widened to FP64 and every product and
// sum is FP64.  R1 may be block-major (bs1 > 0): column c of row i at
// R1[(c / ld1) * bs1 + i * ld1 + c % ld1], blocks of ld1 columns (an even number) bs1
// elements apart (the basis S stored as its blocks S_0, S_1, ...), so a load of two
// columns stays inside a block.
template <typename T1>
struct SrcT {
    const double *L;
    long ldl;
    int kl;
    const T1 *R1;
    long ld1;
    int kr1;
    const double *R2;
    long ld2;
    int kr2;
    long bs1;
};

// offset of column c of R1 from its row start
template <typename T1>
__device__ __forceinline__ long r1_col(const SrcT<T1> &s, int c)
{
    return s.bs1 ? (long)(c / s.ld1) * s.bs1 + c % s.ld1 : (long)c;
}

// 64 consecutive outputs per block; wave w sums chunk partials x in
// [w*gx/4, (w+1)*gx/4) in order, then the four wave sums are added in wave order.
// 32 loads (16 or 8 for what is left of them) are in flight ahead of their additions: a wave's
// share is otherwise a chain of memory latencies.  2000 rows of 16 + 4 columns:
// 3.1 -> 2.7 us with 8 instead of 32 where those do, and with scalar bounds.
__global__ __launch_bounds__(256) void gram_reduce_kernel(const double *__restrict__ part, int gx,
                                                          int kl, int kr1, int kr2, int kl_pad,
                                                          int kr_pad, double *__restrict__ G1,
                                                          double *__restrict__ G2)
{
    constexpr int W = 4;
    __shared__ double red[W][64];
    const int kr = kr1 + kr2;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const long e = (long)blockIdx.x * 64 + lane;
    const bool ok = e < (long)kl * kr;
    const int a = ok ? (int)(e / kr) : 0, b = ok ? (int)(e % kr) : 0;
    const long stride = (long)kl_pad * kr_pad;
    const double *p = part + (long)a * kr_pad + b;
    const int q = (gx + W - 1) / W;
    const int x0 = wave * q, x1 = (x0 + q) < gx ? (x0 + q) : gx;
    double acc = 0.0;
    // past the share's end: its last partial is read again and not added
    auto batch = [&](auto B, int x) {
        constexpr int LD = decltype(B)::value;
        double v[LD];
#pragma unroll
        for (int u = 0; u < LD; u++)
            v[u] = p[(x + u < x1 ? x + u : x1 - 1) * stride];
#pragma unroll
        for (int u = 0; u < LD; u++)
            if (x + u < x1)
                acc += v[u];
    };
    if (ok) {
        int x = x0;
        for (; x1 - x > 16; x += 32)
            batch(std::integral_constant<int, 32>(), x);
        if (x1 - x > 8)
            batch(std::integral_constant<int, 16>(), x);
        else if (x < x1)
            batch(std::integral_constant<int, 8>(), x);
    }
    red[wave][lane] = acc;
    __syncthreads();
    if (wave == 0 && ok) {
        const double sum = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
        if (b < kr1)
            G1[(long)a * kr1 + b] = sum;
        else
            G2[(long)a * kr2 + (b - kr1)] = sum;
    }
}

// The same sums for a small G (kl, k <= 8) and the solve that follows it, in one
// workgroup: up to 8 x 8 the two launches cost more than their work (16 x 16: 12.6 us in one
// workgroup, as much as the two).
// G1 (kl x kr1) and G2 (kl x kr2) are written as above.  factor: x = G1^{-1} G2 (kr1 =
// kl, k = kr2), the factor of G1 kept in lu; otherwise x = (the G1 in lu)^{-1} G1 (k =
// kr1).  Every element receives the same operations in the same order as in
// lu_factor_body and the substitutions of lu.hip: subtractions in ascending order
// of the pivot, the reciprocal pivot last, the backward substitution by
// descending pivot.  Thread (i, j) of 8 x 16 keeps element j of row i: columns
// 0 .. kl - 1 the matrix, 8 .. 8 + k - 1 the right-hand sides.
// 16,384 rows, sm = 4, m = 1: reduce and solve 3.4 + 4.7 us and a launch -> 4.0 us.
constexpr int GS_N = 8;

__global__ __launch_bounds__(1024) void gram_solve_kernel(const double *__restrict__ part, int gx,
                                                          int kl, int kr1, int kr2, int kl_pad,
                                                          int kr_pad, double *__restrict__ G1,
                                                          double *__restrict__ G2,
                                                          double *__restrict__ lu,
                                                          double *__restrict__ x, int *flag,
                                                          int factor)
{
    constexpr int W = 4, LD = 32;
    __shared__ double red[4 * W][64];
    __shared__ double M[GS_N][2 * GS_N + 1];
    const int kr = kr1 + kr2, t = threadIdx.x;
    const int wave = t >> 6, lane = t & 63;
    const int grp = wave / W, wq = wave % W;   // 64 entries to 4 waves, 4 such groups
    if (!factor && t < kl * kl)
        M[t / kl][t % kl] = lu[t];
    for (int e0 = 0; e0 < kl * kr; e0 += 4 * 64) {
        const int e = e0 + grp * 64 + lane;
        const bool ok = e < kl * kr;
        const int a = ok ? e / kr : 0, b = ok ? e % kr : 0;
        const long stride = (long)kl_pad * kr_pad;
        const double *p = part + (long)a * kr_pad + b;
        const int q = (gx + W - 1) / W;
        const int x0 = wq * q, x1 = (x0 + q) < gx ? (x0 + q) : gx;
        double acc = 0.0;
        if (ok) {
            for (int c = x0; c < x1; c += LD) {
                double v[LD];
#pragma unroll
                for (int u = 0; u < LD; u++)
                    v[u] = c + u < x1 ? p[(c + u) * stride] : 0.0;
#pragma unroll
                for (int u = 0; u < LD; u++)
                    if (c + u < x1)
                        acc += v[u];
            }
        }
        red[wave][lane] = acc;
        __syncthreads();
        if (wq == 0 && ok) {
            const double sum =
                ((red[wave][lane] + red[wave + 1][lane]) + red[wave + 2][lane]) + red[wave + 3][lane];
            if (b < kr1) {
                G1[(long)a * kr1 + b] = sum;
                M[a][factor ? b : GS_N + b] = sum;
            } else {
                G2[(long)a * kr2 + (b - kr1)] = sum;
                M[a][GS_N + b - kr1] = sum;
            }
        }
        __syncthreads();
    }
    const int i = t / (2 * GS_N), j = t % (2 * GS_N), k = factor ? kr2 : kr1;
    const bool in = i < kl && (j < GS_N ? j < kl : j - GS_N < k);
    const bool rhs = j >= GS_N;
    double v = in ? M[i][j] : 0.0;
    for (int p = 0; p < kl; p++) {
        // every lane its own: u = M[p][j] / pivot, then M[i][j] -= M[i][p] u
        const double piv = M[p][p], inv = 1.0 / piv;
        const bool col = in && (rhs || (factor && j > p));
        const double u = col ? mul_rn(M[p][j], inv) : 0.0;
        if (col && i == p)
            v = u;
        else if (col && i > p)
            v = sub_rn(v, mul_rn(M[i][p], u));
        if (t == 0 && factor && !(piv != 0.0 && isfinite(piv)))
            *flag = 1;
        __syncthreads();
        if (col && i >= p)
            M[i][j] = v;
        __syncthreads();
    }
    if (factor && in && !rhs)
        lu[i * kl + j] = v;
    for (int q = kl - 1; q > 0; q--) {
        if (in && rhs && i < q) {
            v = sub_rn(v, mul_rn(M[q][j], M[i][q]));
            if (i == q - 1)
                M[i][j] = v;
        }
        __syncthreads();
    }
    if (in && rhs)
        x[(long)i * k + j - GS_N] = v;
}

// 128 columns of L against 128 or 144 of [R1 | R2] (even column counts, 16-byte aligned
// rows).  A stage is 16 rows; the waves load it cooperatively with 16-byte loads, two
// stages ahead, holding the data in registers; the stage is then written to one of
// two LDS buffers and every wave reads its MFMA operands from there, so each row is
// read from HBM once per workgroup.  12 waves of 2 x 3 tiles (144 columns) or 16 of 2 x
// 2 (128) cover all of G; each tile takes its k-steps of 4 rows in row order.
//
// FULL (FP64, every column of the tiles present: 128 x 128 and 128 x 144): the stage
// loop without a bound, a select or an address computation beside one addition per
// load; LDS strides and buffers are immediate offsets.  Every vector instruction
// there is paid in matrix-core time (FP64 MFMAs leave the SIMD few issue slots: 60 more
// of them a stage had cost 2 to 10%).  2,097,152 rows: 128 x 144 1390 -> 1246 us (62
// TFLOP/s), 128 x 128 1249 -> 1110 us.
template <typename T1, int NW, bool FULL>
__global__ __launch_bounds__(NW * 64) void gram_lds_kernel(int n, SrcT<T1> s,
                                                           double *__restrict__ part, int chunk)
{
    constexpr int SR = 16, LDG = 2, MT = 2, NT = NW == 12 ? 3 : 2, GN = NW == 12 ? 3 : 4;
    constexpr int VPT = NW == 12 ? 3 : 2, NTH = NW * 64, KR = NW == 12 ? 144 : 128;
    extern __shared__ double lds[];
    const int kr = s.kr1 + s.kr2;
    const int LDP = lds_row_stride(s.kl), RDP = lds_row_stride(kr);  // padded LDS row strides
    const int BUF = SR * (LDP + RDP);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int lr = lane >> 4, lc = lane & 15;
    const int gm = wave / GN, gn = wave % GN;
    const int ca0 = gm * MT * 16 + lc, cb0 = gn * NT * 16 + lc;

    const int r0 = blockIdx.x * chunk;
    int r1 = r0 + chunk;
    if (r1 > n)
        r1 = n;
    const int nstage = (r1 - r0 + SR - 1) / SR;

    // this lane's share of a stage: 16-byte vector u -> (source row-0 address,
    // row stride in bytes, stage row, LDS offset, FP32 source); an FP32 vector
    // carries 4 columns and is widened into 4 doubles of LDS
    constexpr int E1 = 16 / sizeof(T1);
    const int vl = SR * s.kl / 2, v1 = SR * s.kr1 / E1, v2 = SR * s.kr2 / 2;
    const char *src[VPT];
    long ldb[VPT];
    int srow[VPT], loff[VPT];
    bool isf[VPT];
#pragma unroll
    for (int u = 0; u < VPT; u++) {
        int v = threadIdx.x + NTH * u;
        srow[u] = -1;
        src[u] = reinterpret_cast<const char *>(s.L);
        ldb[u] = 0;
        loff[u] = 0;
        isf[u] = false;
        if (v < vl) {
            const int row = v / (s.kl / 2), c = 2 * (v % (s.kl / 2));
            src[u] = reinterpret_cast<const char *>(s.L + c);
            ldb[u] = s.ldl * (long)sizeof(double);
            srow[u] = row;
            loff[u] = row * LDP + c;
        } else if ((v -= vl) < v1) {
            const int row = v / (s.kr1 / E1), c = E1 * (v % (s.kr1 / E1));
            src[u] = reinterpret_cast<const char *>(s.R1 + r1_col(s, c));
            ldb[u] = s.ld1 * (long)sizeof(T1);
            srow[u] = row;
            loff[u] = SR * LDP + row * RDP + c;
            isf[u] = sizeof(T1) == 4;
        } else if ((v -= v1) < v2) {
            const int row = v / (s.kr2 / 2), c = 2 * (v % (s.kr2 / 2));
            src[u] = reinterpret_cast<const char *>(s.R2 + c);
            ldb[u] = s.ld2 * (long)sizeof(double);
            srow[u] = row;
            loff[u] = SR * LDP + row * RDP + s.kr1 + c;
        }
    }
    uint4 stg[LDG][VPT];
    auto gload = [&](int slot, int st) {
        const int rb = r0 + st * SR;
#pragma unroll
        for (int u = 0; u < VPT; u++) {
            const int row = rb + srow[u];
            const bool ok = srow[u] >= 0 && st < nstage && row < r1;
            stg[slot][u] = ok ? *reinterpret_cast<const uint4 *>(src[u] + (long)row * ldb[u])
                              : uint4{0u, 0u, 0u, 0u};
        }
    };
    auto lstore = [&](int slot, int buf) {
        double *b = lds + buf * BUF;
#pragma unroll
        for (int u = 0; u < VPT; u++) {
            if (srow[u] < 0)
                continue;
            const uint4 w = stg[slot][u];
            if (sizeof(T1) == 4 && isf[u]) {
                float4 f;
                __builtin_memcpy(&f, &w, 16);
                *reinterpret_cast<double2 *>(b + loff[u]) = double2{(double)f.x, (double)f.y};
                *reinterpret_cast<double2 *>(b + loff[u] + 2) = double2{(double)f.z, (double)f.w};
            } else {
                double2 d;
                __builtin_memcpy(&d, &w, 16);
                *reinterpret_cast<double2 *>(b + loff[u]) = d;
            }
        }
    };

    dbl4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
            acc[i][j] = dbl4{0.0, 0.0, 0.0, 0.0};
    // the operands of k-step ks + 1 are read while the MFMAs of ks run (two register sets;
    // the scheduling barriers keep the reads ahead, which the compiler otherwise places
    // just before their MFMAs and waits on)
    auto compute = [&](int buf) {
        const double *bl = lds + buf * BUF;
        const double *br = bl + SR * LDP;
        double av[2][MT], bv[2][NT];
        auto operands = [&](int ks, int p) {
            const int row = ks * 4 + lr;
#pragma unroll
            for (int t = 0; t < MT; t++) {
                const int a = ca0 + 16 * t;
                av[p][t] = a < s.kl ? bl[row * LDP + a] : 0.0;
            }
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const int b = cb0 + 16 * t;
                bv[p][t] = b < kr ? br[row * RDP + b] : 0.0;
            }
        };
        operands(0, 0);
#pragma unroll
        for (int ks = 0; ks < SR / 4; ks++) {
            if (ks + 1 < SR / 4)
                operands(ks + 1, (ks + 1) & 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < NT; j++)
                    acc[i][j] = mfma16x16x4(av[ks & 1][i], bv[ks & 1][j], acc[i][j]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // prologue: stages 0 .. LDG-1 in flight, stage 0 in LDS buffer 0
#pragma unroll
    for (int q = 0; q < LDG; q++)
        gload(q, q);
    lstore(0, 0);
    gload(0, LDG);
    __syncthreads();
    int first = 0;   // first stage of the general loop below
    if constexpr (FULL) {
        constexpr int P = 144, B = SR * 2 * P;   // LDS row stride of 128 and of 144 columns; a buffer
        constexpr int VEC16 = SR * (128 + KR) / 2;   // vectors of a stage
        const int full = (r1 - r0) / SR;
        const char *ptr[VPT];
        long inc[VPT];
        double *dst[VPT];
        bool has[VPT];   // of the whole wave
#pragma unroll
        for (int u = 0; u < VPT; u++) {
            ptr[u] = src[u] + (long)(r0 + (LDG + 1) * SR + max(srow[u], 0)) * ldb[u];
            inc[u] = SR * ldb[u];
            dst[u] = lds + loff[u];
            has[u] = __builtin_amdgcn_readfirstlane(srow[u]) >= 0;
        }
        const double *const bl = lds + lr * P + ca0, *const br = lds + SR * P + lr * P + cb0;
        double av[2][MT], bv[2][NT];
        auto operands = [&](int buf, int ks, int p) {
#pragma unroll
            for (int t = 0; t < MT; t++)
                av[p][t] = bl[buf * B + ks * 4 * P + 16 * t];
#pragma unroll
            for (int t = 0; t < NT; t++)
                bv[p][t] = br[buf * B + ks * 4 * P + 16 * t];
        };
        // loads reach LDG + 1 stages past the one computed
        for (; first + 2 * LDG < full; first += 2) {
#pragma unroll
            for (int q = 0; q < 2; q++) {
                operands(q, 0, 0);
#pragma unroll
                for (int ks = 0; ks < SR / 4; ks++) {
                    if (ks + 1 < SR / 4)
                        operands(q, ks + 1, (ks + 1) & 1);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int i = 0; i < MT; i++)
#pragma unroll
                        for (int j = 0; j < NT; j++)
                            acc[i][j] = mfma16x16x4(av[ks & 1][i], bv[ks & 1][j], acc[i][j]);
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int u = 0; u < VPT; u++)
                    if ((u + 1) * NTH <= VEC16 || has[u]) {
                        double2 d;
                        __builtin_memcpy(&d, &stg[q ^ 1][u], 16);
                        *reinterpret_cast<double2 *>(dst[u] + (q ^ 1) * B) = d;
                        stg[q ^ 1][u] = *reinterpret_cast<const uint4 *>(ptr[u]);
                        ptr[u] += inc[u];
                    }
                __syncthreads();
            }
        }
    }
    // stage st: computed from buffer st & 1; its successor st + 1 sits in
    // register slot (st + 1) % LDG and is stored to the other buffer
    for (int st0 = first; st0 < nstage; st0 += LDG) {
#pragma unroll
        for (int q = 0; q < LDG; q++) {
            const int st = st0 + q;
            if (st < nstage) {
                compute(st & 1);
                const int nslot = (q + 1) % LDG;
                lstore(nslot, (st + 1) & 1);
                gload(nslot, st + 1 + LDG);
            }
            __syncthreads();
        }
    }

    double *out = part + (long)blockIdx.x * 128 * KR;
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                out[(long)((gm * MT + i) * 16 + lr + 4 * r) * KR + (gn * NT + j) * 16 + lc] = acc[i][j][r];
}

// the shapes of gram_lds_kernel: returns 1 when launched
template <typename T1>
int launch_gram_wide(int n, const SrcT<T1> &s, const GramPlan &p, double *work, bool aligned,
                     hipStream_t st)
{
    const int kr = s.kr1 + s.kr2;
    if (!aligned || p.TM != 8 || (p.TN != 8 && p.TN != 9))
        return 0;
    const size_t shm = 2 * 16 * (size_t)(lds_row_stride(s.kl) + lds_row_stride(kr)) * sizeof(double);
    // every column of the tiles present
    const bool full = sizeof(T1) == 8 && s.kl == 128 && kr == p.TN * 16;
#define CACG_GW(NW, FULL)                                                                         \
    do {                                                                                          \
        cacg_allow_lds(gram_lds_kernel<T1, NW, FULL>, shm);                                       \
        hipLaunchKernelGGL((gram_lds_kernel<T1, NW, FULL>), dim3(p.gx), dim3(NW * 64), shm, st, n, s, \
                           work, p.chunk);                                                        \
    } while (0)
    if constexpr (sizeof(T1) == 8) {
        if (full) {
            if (p.TN == 9)
                CACG_GW(12, true);
            else
                CACG_GW(16, true);
            return 1;
        }
    }
    if (p.TN == 9)
        CACG_GW(12, false);
    else
        CACG_GW(16, false);
#undef CACG_GW
    return 1;
}

// ---- few rows of narrow blocks --------------------------------------------------
//
// At most 32 columns of L against 64: a chunk is a few MFMA steps, so a launch is latency
// and what a stage costs beside its loads (the address setup, LDS, a barrier) is most of
// it.  Waves feed the MFMAs from memory: wave (g, ks) forms tile row g against all NT
// column tiles over every fourth step of 4 rows, 4 steps in flight, and the four partial
// sums of a tile row are added in order.  Columns past the last are clamped to it (they
// feed padding only), rows past the last are zeros.
//
// Up to 262,144 rows, 131,072 with an FP32 R1 (the tile kernel against this one, Gram in
// us): 32 + 8 columns 2000 rows 7.8 / 7.1, 20,000 12.3 / 10.7, 250,047 39.5 / 39.0, 500,000
// 65 / 74; 4 + 1 columns 20,000 8.6 / 7.0, 250,047 16.0 / 15.1, 500,000 19 / 21; 16 + 4 columns
// 250,047 22.9 / 21.6, 1,000,000 52 / 59; 24 columns FP32 160,000 28.3 / 27.6, 250,047 35.5 / 37.0.
constexpr int GD_TM = 2, GD_TN = 4;

template <typename T1, int NT>
__global__ __launch_bounds__(256 * GD_TM) void gram_direct_kernel(int n, SrcT<T1> s,
                                                                  double *__restrict__ part,
                                                                  int kr_pad, int chunk)
{
    constexpr int D = 4, PER = NT * 4;
    __shared__ double red[GD_TM][3][PER][64];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int lr = lane >> 4, lc = lane & 15, g = wave >> 2, ks = wave & 3;
    const int r0 = blockIdx.x * chunk, rows = n - r0 < chunk ? n - r0 : chunk;
    const int kr = s.kr1 + s.kr2;
    const double *pa = s.L + (long)r0 * s.ldl + min(16 * g + lc, s.kl - 1);
    const char *pb[NT];
    long ib[NT];
    bool f32[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) {
        const int b = min(16 * j + lc, kr - 1);
        f32[j] = sizeof(T1) == 4 && b < s.kr1;
        ib[j] = b < s.kr1 ? s.ld1 * (long)sizeof(T1) : s.ld2 * (long)sizeof(double);
        pb[j] = b < s.kr1 ? reinterpret_cast<const char *>(s.R1 + r1_col(s, b))
                          : reinterpret_cast<const char *>(s.R2 + (b - s.kr1));
        pb[j] += r0 * ib[j];
    }
    dbl4 acc[NT];
#pragma unroll
    for (int j = 0; j < NT; j++)
        acc[j] = dbl4{0.0, 0.0, 0.0, 0.0};
    double va[2][D], vb[2][D][NT];
    auto load = [&](int p, int k0) {
#pragma unroll
        for (int d = 0; d < D; d++) {
            const int row = k0 + 16 * d + 4 * ks + lr;
            const long i = row < rows ? row : rows - 1;
            const double a = pa[i * s.ldl];
            va[p][d] = row < rows ? a : 0.0;
#pragma unroll
            for (int j = 0; j < NT; j++) {
                const char *q = pb[j] + i * ib[j];
                const double b = f32[j] ? (double)*reinterpret_cast<const float *>(q)
                                        : *reinterpret_cast<const double *>(q);
                vb[p][d][j] = row < rows ? b : 0.0;
            }
        }
    };
    auto compute = [&](int p) {
#pragma unroll
        for (int d = 0; d < D; d++)
#pragma unroll
            for (int j = 0; j < NT; j++)
                acc[j] = mfma16x16x4(va[p][d], vb[p][d][j], acc[j]);
    };
    if (rows > 0)
        load(0, 0);
    for (int k0 = 0; k0 < rows; k0 += 32 * D) {
        if (k0 + 16 * D < rows)
            load(1, k0 + 16 * D);
        compute(0);
        if (k0 + 16 * D >= rows)
            break;
        if (k0 + 32 * D < rows)
            load(0, k0 + 32 * D);
        compute(1);
    }
    if (ks > 0) {
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                red[g][ks - 1][j * 4 + r][lane] = acc[j][r];
    }
    __syncthreads();
    if (ks > 0)
        return;
    double *out = part + (long)blockIdx.x * (blockDim.x / 256 * 16) * kr_pad;
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            double v = acc[j][r];
#pragma unroll
            for (int q = 0; q < 3; q++)
                v += red[g][q][j * 4 + r][lane];
            out[(long)(16 * g + lr + 4 * r) * kr_pad + 16 * j + lc] = v;
        }
}

// launched: 1
template <typename T1>
int launch_gram_direct(int n, const SrcT<T1> &s, const GramPlan &p, double *work, hipStream_t st)
{
    if (n < 1 || n > (sizeof(T1) == 4 ? 1 << 17 : 1 << 18) || p.TM > GD_TM || p.TN > GD_TN)
        return 0;
#define CACG_GD(NT)                                                                               \
    case NT:                                                                                      \
        hipLaunchKernelGGL((gram_direct_kernel<T1, NT>), dim3(p.gx), dim3(256 * p.TM), 0, st, n,  \
                           s, work, p.TN * 16, p.chunk);                                          \
        return 1;
    switch (p.TN) {
        CACG_GD(1)
        CACG_GD(2)
        CACG_GD(3)
        CACG_GD(4)
    default: return 0;
    }
#undef CACG_GD
}

// ---- every other shape: waves share tiles out by group and by rows ----------------
//
// G is cut into blocks of at most 8 x 10 tiles of 16 x 16 (blockIdx.y); a workgroup
// forms one block over one row chunk.  Its waves are NG groups of MT x NT tiles,
// times KS shares of the rows: a stage is 16 KS rows, wave (g, ks) takes every
// KS-th step of 4 rows of it for group g, and the KS partial sums are added in
// order at the end.  Narrow blocks so get as many waves, and as many bytes
// in flight, as wide ones.  Stages are loaded cooperatively two ahead (VEC
// columns a load: 2, or 1 where a source has a single column) and read from one of two
// LDS buffers as in gram_lds_kernel.
// Bound by memory up to about 64 columns, by the matrix cores above.

// two columns, aligned as one
typedef double pair64 __attribute__((ext_vector_type(2), aligned(8)));
typedef float pair32 __attribute__((ext_vector_type(2), aligned(4)));

template <typename T1, int MT, int NT, int VEC, int W, bool ONE>
__global__ __launch_bounds__(64 * W) void gram_tile_kernel(int n, SrcT<T1> s,
                                                         double *__restrict__ part, int kl_pad,
                                                         int kr_pad, int chunk, GramTile g)
{
    constexpr int LDG = 2, VPT = gt_loads(W, VEC);
    using V = typename std::conditional<VEC == 2, pair64, double>::type;
    using V4 = typename std::conditional<VEC == 2, pair32, float>::type;
    constexpr bool one = VEC == 2 && ONE;   // R2 is a single column
    extern __shared__ double lds[];
    const int ca = (int)blockIdx.y / g.nbn * g.TMB * 16, cb = (int)blockIdx.y % g.nbn * g.TNB * 16;
    const int krt = s.kr1 + s.kr2;
    const int kl = s.kl - ca < g.TMB * 16 ? s.kl - ca : g.TMB * 16;
    const int kr = krt - cb < g.TNB * 16 ? krt - cb : g.TNB * 16;
    // R1's columns of the block, then R2's
    const int k1 = s.kr1 - cb < 0 ? 0 : s.kr1 - cb < kr ? s.kr1 - cb : kr, k2 = kr - k1;
    const GtStage<VEC, one, sizeof(T1) == 4> sv(16 * g.KS, kl, k1, k2);
    const int SR = sv.SR, LDP = sv.LDP, RDP = sv.RDP;
    // a tile past the last column reads into the next row (past the last row: 32
    // doubles more); it feeds outputs of the padding only
    const int BUF = SR * (LDP + RDP) + 32;
    const int t = threadIdx.x, nth = blockDim.x;
    const int wave = t >> 6, lane = t & 63, lr = lane >> 4, lc = lane & 15;
    const int gi = wave % g.NG, ks = wave / g.NG;
    const int tm = gi / g.GN * MT, tn = gi % g.GN * NT;
    const int r0 = blockIdx.x * chunk, r1 = n - r0 < chunk ? n : r0 + chunk;
    const int nstage = (r1 - r0 + SR - 1) / SR;

    // this lane's vectors of a stage: source address, and LDS offset, source and row packed
    const char *src[VPT];
    unsigned info[VPT];
    // narrow blocks (one or two tiles a wave, up to 8 waves) need few of the VPT loads: the
    // rest is passed over by scalar branches (2,097,152 rows, 1 + 1 columns: 90 -> 41 us).
    // Others need most, and the branches cost them 5%.
    constexpr bool FEW = MT * NT <= 2 && (W == 8 || sizeof(T1) == 4);
    const int nvec = sv.count();
    auto none = [&](int u) { return FEW && nth * u >= nvec; };
#pragma unroll
    for (int u = 0; u < VPT; u++) {
        info[u] = ~0u;
        src[u] = reinterpret_cast<const char *>(s.L);
        if (none(u))
            continue;
        int c;
        info[u] = sv.vector(t + nth * u, c);
        const long row = r0 + gt_row(info[u]);
        if (info[u] != ~0u)
            src[u] = gt_kind(info[u]) == 0 ? reinterpret_cast<const char *>(s.L + row * s.ldl + ca + c)
                     : gt_kind(info[u]) == 1
                         ? reinterpret_cast<const char *>(s.R1 + row * s.ld1 + r1_col(s, cb + c))
                         : reinterpret_cast<const char *>(s.R2 + row * s.ld2 + cb + c - s.kr1);
    }
    const long incl = (long)SR * s.ldl * sizeof(double), inc1 = (long)SR * s.ld1 * sizeof(T1),
               inc2 = (long)SR * s.ld2 * sizeof(double);
    V stg[LDG][VPT];
    // a single column of R2 has a load of its own, row t of the stage
    double stg1[LDG];
    const double *src1 = s.R2 + (long)(r0 + t) * s.ld2;
    auto gload = [&](int slot, int st) {
        const int left = gt_stage_rows(r1 - r0, SR, st);
        if constexpr (one) {
            stg1[slot] = t < left && k2 > 0 ? *src1 : 0.0;
            src1 += SR * s.ld2;
        }
#pragma unroll
        for (int u = 0; u < VPT; u++) {
            if (none(u))
                break;
            const int kind = gt_kind(info[u]);
            V w{};
            if (gt_row(info[u]) < left) {
                if (sizeof(T1) == 4 && kind == 1) {
                    const V4 f = *reinterpret_cast<const V4 *>(src[u]);
                    __builtin_memcpy(&w, &f, sizeof(f));
                } else {
                    w = *reinterpret_cast<const V *>(src[u]);
                }
            }
            stg[slot][u] = w;
            src[u] += kind == 0 ? incl : kind == 1 ? inc1 : inc2;
        }
    };
    auto lstore = [&](int slot, int buf) {
        double *b = lds + buf * BUF;
        if constexpr (one) {
            if (t < SR && k2 > 0)
                b[SR * LDP + t * RDP + k1] = stg1[slot];
        }
#pragma unroll
        for (int u = 0; u < VPT; u++) {
            if (none(u))
                break;
            if (info[u] == ~0u)
                continue;
            V w = stg[slot][u];
            if (sizeof(T1) == 4 && gt_kind(info[u]) == 1) {
                V4 f;
                __builtin_memcpy(&f, &w, sizeof(f));
                if constexpr (VEC == 2)
                    w = V{(double)f.x, (double)f.y};
                else
                    w = (double)f;
            }
            *reinterpret_cast<V *>(b + (info[u] >> 12)) = w;
        }
    };
    dbl4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
            acc[i][j] = dbl4{0.0, 0.0, 0.0, 0.0};
    auto compute = [&](int buf) {
        const double *bl = lds + buf * BUF + (4 * ks + lr) * LDP + tm * 16 + lc;
        const double *br = lds + buf * BUF + SR * LDP + (4 * ks + lr) * RDP + tn * 16 + lc;
        double av[2][MT], bv[2][NT];
        auto operands = [&](int q, int p) {
#pragma unroll
            for (int i = 0; i < MT; i++)
                av[p][i] = bl[4 * q * g.KS * LDP + 16 * i];
#pragma unroll
            for (int j = 0; j < NT; j++)
                bv[p][j] = br[4 * q * g.KS * RDP + 16 * j];
        };
        operands(0, 0);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            if (q + 1 < 4)
                operands(q + 1, (q + 1) & 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < NT; j++)
                    acc[i][j] = mfma16x16x4(av[q & 1][i], bv[q & 1][j], acc[i][j]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
#pragma unroll
    for (int q = 0; q < LDG; q++)
        gload(q, q);
    lstore(0, 0);
    gload(0, LDG);
    __syncthreads();
    // whole stages without row tests or selects, as in gram_lds_kernel: an addition per
    // load, and lanes without a vector load the start of L and store nothing.  Not where
    // 16 waves' 128 registers would spill more (2 x 3, 1 x 4 and 1 x 5 tiles keep a few
    // registers in scratch as they are), nor for one or two tiles a wave, which are
    // bound by memory (2,097,152 rows of 16 + 4 columns: 112 -> 118 us).  300,000 rows of 96
    // columns 124 -> 113 us, 1,000,000 of 64 + 8 240 -> 222 us, 300,000 of 99 + 11 184 -> 168.
    int first = 0;
    const int full = (r1 - r0) / SR;
    if (sizeof(T1) == 8 && VEC == 2 && MT * NT >= 3 && (W == 8 || MT * NT <= 4) && full > 2 * LDG) {
        long inc[VPT];
        V *dst[VPT];
#pragma unroll
        for (int u = 0; u < VPT; u++) {
            const int kind = gt_kind(info[u]);
            inc[u] = info[u] == ~0u ? 0 : kind == 0 ? incl : kind == 1 ? inc1 : inc2;
            dst[u] = reinterpret_cast<V *>(lds + (info[u] >> 12));
            if (info[u] == ~0u)
                src[u] = reinterpret_cast<const char *>(s.L);
        }
        for (; first + 2 * LDG < full; first += 2) {
#pragma unroll
            for (int q = 0; q < 2; q++) {
                compute(q);
#pragma unroll
                for (int u = 0; u < VPT; u++) {
                    if (info[u] != ~0u)
                        *reinterpret_cast<V *>(reinterpret_cast<double *>(dst[u]) + (q ^ 1) * BUF) =
                            stg[q ^ 1][u];
                    stg[q ^ 1][u] = *reinterpret_cast<const V *>(src[u]);
                    src[u] += inc[u];
                }
                __syncthreads();
            }
        }
    }
    for (int st0 = first; st0 < nstage; st0 += LDG) {
#pragma unroll
        for (int q = 0; q < LDG; q++) {
            const int st = st0 + q;
            if (st < nstage) {
                compute(st & 1);
                const int nslot = (q + 1) % LDG;
                lstore(nslot, (st + 1) & 1);
                gload(nslot, st + 1 + LDG);
            }
            __syncthreads();
        }
    }
    // the KS shares of a group, added in order
    if (g.KS > 1) {
        constexpr int per = MT * NT * 4;
        double *dst = lds + ((ks - 1) * g.NG + gi) * per * 64 + lane;
        if (ks > 0) {
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < NT; j++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        dst[((i * NT + j) * 4 + r) * 64] = acc[i][j][r];
        }
        __syncthreads();
        if (ks > 0)
            return;
        for (int q = 0; q + 1 < g.KS; q++) {
            const double *from = lds + (q * g.NG + gi) * per * 64 + lane;
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < NT; j++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        acc[i][j][r] += from[((i * NT + j) * 4 + r) * 64];
        }
    }
    double *out = part + (long)blockIdx.x * kl_pad * kr_pad;
#pragma unroll
    for (int i = 0; i < MT; i++) {
        const int a = ca + (tm + i) * 16;
        if (tm + i >= g.TMB || a >= kl_pad)
            continue;
#pragma unroll
        for (int j = 0; j < NT; j++) {
            const int b = cb + (tn + j) * 16;
            if (tn + j >= g.TNB || b >= kr_pad)
                continue;
#pragma unroll
            for (int r = 0; r < 4; r++)
                out[(long)(a + lr + 4 * r) * kr_pad + b + lc] = acc[i][j][r];
        }
    }
}

template <typename T1, int VEC>
int launch_gram_tile(int n, const SrcT<T1> &s, const GramPlan &p, const GramTile &g, double *work,
                     hipStream_t st)
{
    const int kl_pad = p.TM * 16, kr_pad = p.TN * 16;
    const dim3 grid(p.gx, (p.TM + g.TMB - 1) / g.TMB * g.nbn), block(64 * g.NG * g.KS);
#define CACG_GT(M, N, WV, ONE)                                                                    \
    if (g.MT == M && g.NT == N && g.W == WV) {                                                    \
        cacg_allow_lds(gram_tile_kernel<T1, M, N, VEC, WV, ONE>, g.lds);                          \
        hipLaunchKernelGGL((gram_tile_kernel<T1, M, N, VEC, WV, ONE>), grid, block, g.lds, st, n, \
                           s, work, kl_pad, kr_pad, p.chunk, g);                                  \
        return 0;                                                                                 \
    }
    if constexpr (VEC == 2 && sizeof(T1) == 8) {
        if (s.kr2 == 1) {
            CACG_GT(1, 1, 8, true)
            CACG_GT(1, 1, 16, true)
            CACG_GT(1, 2, 8, true)
            CACG_GT(1, 2, 16, true)
            return (int)hipErrorInvalidValue;
        }
    }
#define CACG_GTW(M, N) CACG_GT(M, N, 8, false) CACG_GT(M, N, 16, false)
    CACG_GTW(1, 1)
    CACG_GTW(1, 2)
    CACG_GTW(1, 3)
    CACG_GTW(1, 4)
    CACG_GTW(1, 5)
    CACG_GTW(2, 2)
    CACG_GTW(2, 3)
#undef CACG_GTW
#undef CACG_GT
    return (int)hipErrorInvalidValue;
}

struct GramSolve {
    double *lu, *x;
    int *flag, factor;
};

template <typename T1>
int gram_fast(int n, const double *L, long ldl, int kl, const T1 *R1, long ld1, int kr1,
              const double *R2, long ld2, int kr2, double *G1, double *G2, double *d_work,
              hipStream_t st, long bs1 = 0, const GramSolve *sol = nullptr)
{
    if (n < 0 || kl <= 0 || kr1 < 0 || kr2 < 0 || kr1 + kr2 <= 0)
        return (int)hipErrorInvalidValue;
    GramPlan p = plan_gram(n, kl, kr1 + kr2);
    tile_chunks(n, p);
    const SrcT<T1> s = {L, ldl, kl, R1, ld1, kr1, R2, ld2, kr2, bs1};
    constexpr int E1 = 16 / sizeof(T1);
    auto al16 = [](const void *q) { return ((uintptr_t)q & 15) == 0; };
    // 16-byte vectors: column counts and row strides in whole vectors, aligned rows
    const bool aligned = p.KS == 1 && kl % 2 == 0 && kr1 % E1 == 0 && kr2 % 2 == 0 &&
                         ldl % 2 == 0 && ld1 % E1 == 0 && bs1 % E1 == 0 &&
                         (kr2 == 0 || ld2 % 2 == 0) && al16(L) && al16(R1) &&
                         (kr2 == 0 || al16(R2));
    // a block-major R1 is taken in the shapes cacg_gram_blk_supported names only
    if (bs1 && !(aligned && blk_shape(p, kl, kr1)))
        return (int)hipErrorInvalidValue;
    if (!launch_gram_direct(n, s, p, d_work, st) &&
        !launch_gram_wide(n, s, p, d_work, aligned, st)) {
        // pairs of columns (16-byte loads need no alignment beyond the element's), or
        // single ones where a source has only one
        constexpr bool f32 = sizeof(T1) == 4;
        GramTile g;
        const int rc =
            plan_pairs(n, kl, kr1, kr2, p, f32, g)
                ? launch_gram_tile<T1, 2>(n, s, p, g, d_work, st)
                : launch_gram_tile<T1, 1>(n, s, p, plan_tile(p.TM, p.TN, 1, p.chunk, p.gx, f32),
                                              d_work, st);
        if (rc)
            return rc;
    }
    CACG_LAUNCH_CHECK();
    if (sol) {
        hipLaunchKernelGGL(gram_solve_kernel, dim3(1), dim3(1024), 0, st, d_work, p.gx, kl, kr1, kr2,
                           p.TM * 16, p.TN * 16, G1, G2, sol->lu, sol->x, sol->flag, sol->factor);
        CACG_LAUNCH_CHECK();
        return 0;
    }
    const long outs = (long)kl * (kr1 + kr2);
    hipLaunchKernelGGL(gram_reduce_kernel, dim3(cacg_grid(outs, 64, 0)), dim3(256), 0, st, d_work,
                       p.gx, kl, kr1, kr2, p.TM * 16, p.TN * 16, G1, G2);
    CACG_LAUNCH_CHECK();
    return 0;
}

}  // namespace

namespace {

template <int NJ>
int launch_gram_ref(int n, const GrefSrc &s, long blocks, int nbb, double *G1, double *G2,
                    hipStream_t st)
{
    constexpr size_t lds = 2 * GrefShape<NJ>::BUF * sizeof(double2);
    cacg_allow_lds(gram_ref_kernel<NJ>, lds);
    hipLaunchKernelGGL(gram_ref_kernel<NJ>, dim3((unsigned)blocks), dim3(512), lds, st, n, s, nbb,
                       G1, G2);
    CACG_LAUNCH_CHECK();
    return 0;
}

}  // namespace

extern "C" int cacg_k_gram_ref(int n, const double *L, long ldl, int kl, const double *R1, long ld1,
                               int kr1, const double *R2, long ld2, int kr2, double *G1,
                               double *G2, hipStream_t st)
{
    if (n < 0 || kl <= 0 || kr1 < 0 || kr2 < 0 || kr1 + kr2 <= 0)
        return (int)hipErrorInvalidValue;
    if (kr2 > 0 && !R2)
        return (int)hipErrorInvalidValue;
    if (n == 0) {
        // empty sums: zero blocks
        int rc = kr1 > 0 ? cacg_k_fill_f64(G1, (long)kl * kr1, 0.0, st) : 0;
        if (!rc && kr2 > 0)
            rc = cacg_k_fill_f64(G2, (long)kl * kr2, 0.0, st);
        return rc;
    }
    const int kr = kr1 + kr2;
    const GrefSrc s = {L, ldl, kl, R1, ld1, kr1, R2, ld2, kr2};
    // the narrowest block whose grid gives no CU a second workgroup: 262,144 rows
    // of 28, 56, 112 and 128 against 144 columns take 1.30, 1.32, 1.50 and 1.70 ms with
    // NJ = 1, 2, 4 and 5
    const int nbb = (kr + 15) / 16;
    const auto blocks = [&](int nj) { return (long)((kl + nj - 1) / nj) * nbb; };
#define CACG_GREF(nj)                                                                             \
    if (blocks(nj) <= 256)                                                                        \
    return launch_gram_ref<nj>(n, s, blocks(nj), nbb, G1, G2, st)
    CACG_GREF(1);
    CACG_GREF(2);
    CACG_GREF(4);
    CACG_GREF(5);
#undef CACG_GREF
    return launch_gram_ref<8>(n, s, blocks(8), nbb, G1, G2, st);
}

extern "C" long cacg_gram_workspace(int kl, int kr)
{
    // upper bound over n: gx <= 512
    return 512L * ((kl + 15) / 16 * 16) * ((kr + 15) / 16 * 16);
}

extern "C" long cacg_gram_workspace_n(int n, int kl, int kr)
{
    if (n <= 0 || kl <= 0 || kr <= 0)
        return 0;
    const GramPlan p = plan_gram(n, kl, kr);
    return (long)p.gx * (p.TM * 16) * (p.TN * 16);
}

extern "C" int cacg_k_gram_fast(int n, const double *L, long ldl, int kl, const double *R1,
                                long ld1, int kr1, const double *R2, long ld2, int kr2, double *G1,
                                double *G2, double *d_work, hipStream_t st)
{
    return gram_fast<double>(n, L, ldl, kl, R1, ld1, kr1, R2, ld2, kr2, G1, G2, d_work, st);
}

extern "C" int cacg_gram_blk_supported(int n, int kl, int kr1, int bw)
{
    if (n <= 0 || kl <= 0 || bw <= 0 || kr1 <= 0 || kr1 % bw != 0 || bw % 2 != 0 || kl % 2 != 0)
        return 0;
    // 16-byte aligned L, R1 and ldl = kl assumed
    return blk_shape(plan_gram(n, kl, kr1), kl, kr1) ? 1 : 0;
}

extern "C" int cacg_k_gram_fast_blk(int n, const double *L, long ldl, int kl, const double *R1,
                                    int bw, long bs, int kr1, double *G1, double *d_work,
                                    hipStream_t st)
{
    if (bw <= 0 || bs < (long)n * bw || kr1 % bw != 0)
        return (int)hipErrorInvalidValue;
    return gram_fast<double>(n, L, ldl, kl, R1, bw, kr1, nullptr, 1, 0, G1, nullptr, d_work, st,
                             bs);
}

extern "C" int cacg_gram_solve_supported(int sm, int m)
{
    return sm >= 1 && sm <= GS_N && m >= 1 && m <= GS_N;
}

extern "C" int cacg_k_gram_alpha(int n, int sm, int m, const double *Q, const double *AQ,
                                 const double *R, double *QtAQ, double *QtR, double *alpha,
                                 double *lu, int *d_flag, double *d_work, hipStream_t st)
{
    if (n <= 0 || !cacg_gram_solve_supported(sm, m))
        return (int)hipErrorInvalidValue;
    const GramSolve sol = {lu, alpha, d_flag, 1};
    return gram_fast<double>(n, Q, sm, sm, AQ, sm, sm, R, m, m, QtAQ, QtR, d_work, st, 0, &sol);
}

extern "C" int cacg_k_gram_beta(int n, int sm, const double *AQ, const double *S, const float *S32,
                                double *QtAS, double *beta, double *lu, double *d_work,
                                hipStream_t st)
{
    if (n <= 0 || !cacg_gram_solve_supported(sm, 1))
        return (int)hipErrorInvalidValue;
    const GramSolve sol = {lu, beta, nullptr, 0};
    if (S32)
        return gram_fast<float>(n, AQ, sm, sm, S32, sm, sm, nullptr, 1, 0, QtAS, nullptr, d_work,
                                st, 0, &sol);
    return gram_fast<double>(n, AQ, sm, sm, S, sm, sm, nullptr, 1, 0, QtAS, nullptr, d_work, st, 0,
                             &sol);
}

extern "C" int cacg_k_gram_fast_f64f32(int n, const double *L, long ldl, int kl, const float *R1,
                                       long ld1, int kr1, const double *R2, long ld2, int kr2,
                                       double *G1, double *G2, double *d_work, hipStream_t st)
{
    return gram_fast<float>(n, L, ldl, kl, R1, ld1, kr1, R2, ld2, kr2, G1, G2, d_work, st);
}
