// Small dense solve x = lhs^{-1} rhs, the reference's LUsolver_v1_KeeplhsMat
// (src/DLSsolvers.c:106-208): Crout factorisation with unit-diagonal U and no
// pivoting, forward then backward substitution.  gfx950.
//
// Every element of the factor and of y = L^{-1} rhs receives its subtractions
// a - l u (product and difference rounded separately) in ascending order of
// the pivot, with the reciprocal pivot applied last, as in the reference's
// loops, so both are the reference's bits however the work is divided.  The
// backward substitution of mode FAST is column-oriented (descending pivot);
// mode REFERENCE keeps the reference's ascending sums.
//
// N <= 128: one workgroup factors (lu_factor_body), panels of 8 pivots in
// the registers of a few waves, the trailing matrix in the registers of all
// 16; up to 32 right-hand sides ride along as further columns, so the forward
// substitution costs no step of its own.  N > 128: blocks of 128, a factor
// kernel, triangular solves and products per block, each over many CUs.
#include <math.h>

#include <type_traits>

#include "kcommon.hpp"

namespace {

constexpr int LU_T = 1024;
constexpr int LU_B = 128;      // rows of a diagonal block
constexpr int LU_P = 8;        // pivots of a panel
constexpr int LU_PS = 10;      // LDS row stride of a panel: 20 words, so 16 lanes' 16-byte
                               // reads of consecutive rows cover all 64 banks
constexpr int LU_K = 32;       // right-hand sides that ride along with a factorisation
constexpr int TRI_W = 8;       // waves of a triangular-solve workgroup

// ---- substitutions of one vector by one wave -------------------------------------
//
// Lane l holds entries l (y0) and 64 + l (y1) of a vector of nb <= 128.  Step q
// finishes entry q, hands it to the wave by readlane, and the other entries
// subtract its multiple.  T(q) points to the multipliers of step q (entry i at
// T(q)[i]; entries outside the triangle are read and not used).  A wave issues
// one FP64 instruction about every 8.5 cycles and an LDS read waits for 64 or
// more, so the multipliers of the next 4 steps are read while the current 4
// run.

// ascending: entry i > q subtracts y_q T(q)[i]; with SCALE entry q is first
// multiplied by its reciprocal pivot (d0, d1: those of this lane's entries)
template <bool SCALE, typename F>
__device__ __forceinline__ void tri_forward(int nb, F T, double d0, double d1, double &y0,
                                            double &y1)
{
    const int l = threadIdx.x & 63;
    const int n0 = nb < 64 ? nb : 64;
    const bool two = nb > 64;
    double a[2][4], b[2][4];
    auto load = [&](int s, int q0, bool lo) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const double *t = T(q0 + u < nb ? q0 + u : nb - 1);
            a[s][u] = lo ? t[l] : 0.0;
            b[s][u] = two ? t[64 + l] : 0.0;
        }
    };
    auto steps0 = [&](int s, int q0) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int q = q0 + u;
            if (q < n0) {
                const double yd = SCALE ? mul_rn(y0, d0) : y0;
                const double yq = readlane_f64(yd, q);
                const double w = sub_rn(y0, mul_rn(yq, a[s][u]));
                y0 = l > q ? w : (SCALE && l == q ? yd : y0);
                if (two)
                    y1 = sub_rn(y1, mul_rn(yq, b[s][u]));
            }
        }
    };
    auto steps1 = [&](int s, int q0) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int q = q0 + u;
            if (q < nb) {
                const double yd = SCALE ? mul_rn(y1, d1) : y1;
                const double yq = readlane_f64(yd, q - 64);
                const double w = sub_rn(y1, mul_rn(yq, b[s][u]));
                y1 = l > q - 64 ? w : (SCALE && l == q - 64 ? yd : y1);
            }
        }
    };
    load(0, 0, true);
#pragma unroll 1
    for (int q0 = 0; q0 < n0; q0 += 8) {
        load(1, q0 + 4, true);
        __builtin_amdgcn_sched_barrier(0);
        steps0(0, q0);
        load(0, q0 + 8, true);
        __builtin_amdgcn_sched_barrier(0);
        steps0(1, q0 + 4);
    }
    if (!two)
        return;
    load(0, 64, false);
#pragma unroll 1
    for (int q0 = 64; q0 < nb; q0 += 8) {
        load(1, q0 + 4, false);
        __builtin_amdgcn_sched_barrier(0);
        steps1(0, q0);
        load(0, q0 + 8, false);
        __builtin_amdgcn_sched_barrier(0);
        steps1(1, q0 + 4);
    }
}

// descending, unit diagonal: entry i < q subtracts y_q T(q)[i]
template <typename F>
__device__ __forceinline__ void tri_backward(int nb, F T, double &y0, double &y1)
{
    const int l = threadIdx.x & 63;
    const int n0 = nb < 64 ? nb : 64;
    double a[2][4], b[2][4];
    auto load = [&](int s, int q0, bool hi) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const double *t = T(q0 - u > 0 ? q0 - u : 0);
            a[s][u] = t[l];
            b[s][u] = hi ? t[64 + l] : 0.0;
        }
    };
    auto steps1 = [&](int s, int q0) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int q = q0 - u;
            if (q >= 64) {
                const double yq = readlane_f64(y1, q - 64);
                const double w = sub_rn(y1, mul_rn(yq, b[s][u]));
                y1 = l < q - 64 ? w : y1;
                y0 = sub_rn(y0, mul_rn(yq, a[s][u]));
            }
        }
    };
    auto steps0 = [&](int s, int q0) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int q = q0 - u;
            if (q > 0) {
                const double yq = readlane_f64(y0, q);
                const double w = sub_rn(y0, mul_rn(yq, a[s][u]));
                y0 = l < q ? w : y0;
            }
        }
    };
    if (nb > 64) {
        load(0, nb - 1, true);
#pragma unroll 1
        for (int q0 = nb - 1; q0 >= 64; q0 -= 8) {
            load(1, q0 - 4, true);
            __builtin_amdgcn_sched_barrier(0);
            steps1(0, q0);
            load(0, q0 - 8, true);
            __builtin_amdgcn_sched_barrier(0);
            steps1(1, q0 - 4);
        }
    }
    load(0, n0 - 1, false);
#pragma unroll 1
    for (int q0 = n0 - 1; q0 > 0; q0 -= 8) {
        load(1, q0 - 4, false);
        __builtin_amdgcn_sched_barrier(0);
        steps0(0, q0);
        load(0, q0 - 8, false);
        __builtin_amdgcn_sched_barrier(0);
        steps0(1, q0 - 4);
    }
}

// ---- factorisation of up to 128 rows ----------------------------------------------

// columns of U above the diagonal, packed: column q at q (q - 1) / 2
__host__ __device__ inline int upk(int q) { return q * (q - 1) / 2; }

// dynamic LDS (doubles) of lu_factor_body: the column panel (128 rows), the row
// panel (128 columns and LU_K right-hand sides), and with `back` the packed U
// and the right-hand sides after the forward substitution
__host__ __device__ inline int lu_factor_lds(int N, int k, bool back)
{
    const int pan = LU_PS * (2 * LU_B + LU_K);
    return back ? pan + upk(N) + 2 * LU_B + k * (N + 1) + LU_B : pan;
}

// Factor the N x N block at lhs (row stride ldl) into gw (row stride ldg; lhs
// may be gw), N <= 128, with k <= LU_K right-hand sides: y = L^{-1} rhs, and
// with back also x = U^{-1} y in mode FAST's order; written to x (N x k).
//
// Lane (tr, tc) of a 32 x 32 grid keeps elements (tr + 32 i, tc + 32 j) and
// right-hand side tc of rows tr + 32 i in registers.  Per panel of 8 pivots:
//   1. the panel's columns (all rows below) and rows (all columns to the right,
//      the right-hand sides among them) lie in LDS.  A row wave holds the 8
//      panel rows and 56 rows below, one row of the panel's 8 columns a lane;
//      a column wave the 8 panel columns and 56 columns to the right, one
//      column of the panel's 8 rows a lane.  Each factors the 8 x 8 diagonal
//      block for itself, passing pivots between lanes by readlane, so l and u
//      of the whole panel are ready without a barrier inside it;
//   2. every lane applies the 8 rank-1 updates to its elements, in order, and
//      the owners of the next panel put it into LDS.
// Three barriers per 8 pivots (panel factored, panel's readers done, next panel in
// place).  What bounds it is the chain of pivots: one
// reciprocal, one product and one subtraction each, about 200 cycles; a barrier
// and a broadcast through LDS for every pivot had taken 1870.
__device__ __forceinline__ void lu_factor_body(int N, const double *lhs, long ldl, double *gw,
                                               long ldg, int k, const double *__restrict__ rhs,
                                               double *__restrict__ x, int *flag, bool back,
                                               double *lds)
{
    double *cp = lds;                            // column panel: row r at cp + r LU_PS
    double *rp = lds + LU_PS * LU_B;             // row panel: column c at rp + c LU_PS
    double *U = lds + LU_PS * (2 * LU_B + LU_K); // packed U
    double *ys = U + upk(N) + 2 * LU_B;          // right-hand side c at ys + c (N + 1)
    const int t = threadIdx.x, tr = t >> 5, tc = t & 31;
    const int wave = t >> 6, lane = t & 63;
    double v[4][4], vr[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int r = tr + 32 * i;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int c = tc + 32 * j;
            v[i][j] = (r < N && c < N) ? lhs[(long)r * ldl + c] : (r == c ? 1.0 : 0.0);
        }
        vr[i] = (r < N && tc < k) ? rhs[(long)r * k + tc] : 0.0;
    }
    auto publish = [&](auto I, int q0) {
        constexpr int ip = decltype(I)::value;
        const int dr = tr - q0, dc = tc - q0;
        if (dr >= 0 && dr < LU_P) {
#pragma unroll
            for (int j = ip; j < 4; j++)
                rp[(tc + 32 * j) * LU_PS + dr] = v[ip][j];
            if (k > 0)
                rp[(LU_B + tc) * LU_PS + dr] = vr[ip];
        }
        if (dc >= 0 && dc < LU_P) {
#pragma unroll
            for (int i = ip; i < 4; i++)
                cp[(tr + 32 * i) * LU_PS + dc] = v[i][ip];
        }
    };
    // elements above or left of the next panel are final and stored: they take
    // part here only because leaving them out would cost a test, and are not
    // read again
    auto update = [&](auto I) {
        constexpr int ip = decltype(I)::value;
#pragma unroll 1
        for (int p = 0; p < LU_P; p += 2) {
            double2 l[4];
#pragma unroll
            for (int i = ip; i < 4; i++)
                l[i] = *(const double2 *)(cp + (tr + 32 * i) * LU_PS + p);
#pragma unroll
            for (int j = ip; j < 4; j++) {
                const double2 u = *(const double2 *)(rp + (tc + 32 * j) * LU_PS + p);
#pragma unroll
                for (int i = ip; i < 4; i++) {
                    v[i][j] = sub_rn(v[i][j], mul_rn(l[i].x, u.x));
                    v[i][j] = sub_rn(v[i][j], mul_rn(l[i].y, u.y));
                }
            }
            if (k > 0) {
                const double2 u = *(const double2 *)(rp + (LU_B + tc) * LU_PS + p);
#pragma unroll
                for (int i = ip; i < 4; i++) {
                    vr[i] = sub_rn(vr[i], mul_rn(l[i].x, u.x));
                    vr[i] = sub_rn(vr[i], mul_rn(l[i].y, u.y));
                }
            }
        }
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;
    publish(I0{}, 0);
    __syncthreads();
#pragma unroll 1
    for (int P0 = 0; P0 < N; P0 += LU_P) {
        const int P1 = P0 + LU_P;
        // ---- 1: the panel
        const int below = N - P1 > 0 ? N - P1 : 0;
        const int nrw = below > 0 ? (below + 55) / 56 : 1;
        const int ncw = (below + k + 55) / 56;
        if (wave < nrw) {
            const int r = lane < LU_P ? P0 + lane : P1 + wave * 56 + lane - LU_P;
            const bool in = r < N;
            double w[LU_P];
#pragma unroll
            for (int j = 0; j < LU_P; j++)
                w[j] = cp[(r < LU_B ? r : 0) * LU_PS + j];
            int bad = 0;
#pragma unroll
            for (int p = 0; p < LU_P; p++) {
                const double piv = readlane_f64(w[p], p);
                if (P0 + p < N && !(piv != 0.0 && isfinite(piv)))
                    bad = 1;
                const double inv = 1.0 / piv;
#pragma unroll
                for (int j = p + 1; j < LU_P; j++) {
                    const double u = mul_rn(readlane_f64(w[j], p), inv);
                    const double d = sub_rn(w[j], mul_rn(w[p], u));
                    w[j] = lane > p ? d : (lane == p ? u : w[j]);
                }
            }
            if (in && (lane >= LU_P || wave == 0)) {
#pragma unroll
                for (int j = 0; j < LU_P; j++) {
                    if (lane >= LU_P)
                        cp[r * LU_PS + j] = w[j];
                    if (P0 + j < N) {
                        gw[(long)r * ldg + P0 + j] = w[j];
                        if (back && lane < j)
                            U[upk(P0 + j) + r] = w[j];
                    }
                }
            }
            if (wave == 0 && lane == 0 && bad)
                *flag = 1;
        } else if (wave < nrw + ncw) {
            // column: the panel's own, one to the right, or a right-hand side
            const int e = (wave - nrw) * 56 + lane - LU_P;
            const int c = lane < LU_P ? P0 + lane : (e < below ? P1 + e : LU_B + e - below);
            const bool rh = lane >= LU_P && e >= below;
            const bool in = lane >= LU_P && e < below + k;
            double w[LU_P];
#pragma unroll
            for (int i = 0; i < LU_P; i++)
                w[i] = rp[(in || lane < LU_P ? c : 0) * LU_PS + i];
#pragma unroll
            for (int p = 0; p < LU_P; p++) {
                const double inv = 1.0 / readlane_f64(w[p], p);
                const double u = mul_rn(w[p], inv);
                w[p] = lane > p ? u : w[p];
#pragma unroll
                for (int i = p + 1; i < LU_P; i++) {
                    const double l = readlane_f64(w[i], p);
                    const double d = sub_rn(w[i], mul_rn(l, u));
                    w[i] = lane > p ? d : w[i];
                }
            }
            if (in) {
#pragma unroll
                for (int i = 0; i < LU_P; i++) {
                    const int r = P0 + i;
                    rp[c * LU_PS + i] = w[i];
                    if (r >= N)
                        continue;
                    if (rh) {
                        if (back)
                            ys[(c - LU_B) * (N + 1) + r] = w[i];
                        else
                            x[(long)r * k + c - LU_B] = w[i];
                    } else {
                        gw[(long)r * ldg + c] = w[i];
                        if (back)
                            U[upk(c) + r] = w[i];
                    }
                }
            }
        }
        __syncthreads();
        if (P1 >= N)
            break;
        // ---- 2: the trailing elements
        switch (P0 / 32) {
        case 0: update(I0{}); break;
        case 1: update(I1{}); break;
        case 2: update(I2{}); break;
        default: update(I3{}); break;
        }
        __syncthreads();   // the panel has been read: the next one may be written
        switch (P1 / 32) {
        case 0: publish(I0{}, P1 % 32); break;
        case 1: publish(I1{}, P1 % 32); break;
        case 2: publish(I2{}, P1 % 32); break;
        default: publish(I3{}, P1 % 32); break;
        }
        __syncthreads();
    }
    if (!back)
        return;
    __syncthreads();
    for (int c = wave; c < k; c += LU_T / 64) {
        double *y = ys + c * (N + 1);
        double y0 = y[lane < N ? lane : 0], y1 = y[64 + lane < N ? 64 + lane : 0];
        tri_backward(N, [&](int q) { return (const double *)(U + upk(q)); }, y0, y1);
        if (lane < N)
            x[(long)lane * k + c] = y0;
        if (64 + lane < N)
            x[(long)(64 + lane) * k + c] = y1;
    }
}

__global__ __launch_bounds__(LU_T) void lu_factor_kernel(int N, const double *lhs, long ldl,
                                                         double *gw, long ldg, int k,
                                                         const double *__restrict__ rhs,
                                                         double *__restrict__ x, int *flag,
                                                         int back)
{
    extern __shared__ double lds[];
    lu_factor_body(N, lhs, ldl, gw, ldg, k, rhs, x, flag, back != 0, lds);
}

// ---- triangular solves with a kept factor block -----------------------------------

// A set of vectors: entry i of vector v at in / out + v vs + i es
struct TriSet {
    const double *in;
    double *out;
    long vs, es;
    int count;
    int kind;
};
enum { TRI_FORWARD = 1, TRI_BACKWARD = 2, TRI_UT = 4 };

__host__ __device__ inline int tri_lds(int nb) { return (nb + 1) * (nb + 1) + LU_B; }

// Vectors first .. of a set, one per wave and step, by the nb x nb factor block at
// F (row stride ldf): kind FORWARD: L y = v; FORWARD | BACKWARD: then U x = y
// (descending pivots); BACKWARD alone: U x = v; UT: y U = v (rows of L left of
// the block: ascending pivots, unit diagonal).  The block is copied to LDS
// first, column by column (UT: row by row) with the odd stride nb + 1, so the
// multipliers of a step lie in consecutive words.
__device__ __forceinline__ void tri_body(int nb, const double *F, long ldf, const TriSet &s,
                                         int first, int step, double *lds)
{
    const int t = threadIdx.x, R = nb + 1;
    const int w = t >> 6, l = t & 63;
    const bool ut = s.kind == TRI_UT;
    // a wave copies rows w, w + TRI_W, ...: 64 columns a load, 8 rows in flight
    for (int r0 = w; r0 < nb; r0 += 8 * TRI_W) {
        double f[8][2];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int r = r0 + u * TRI_W;
            const double *p = F + (long)(r < nb ? r : 0) * ldf;
            f[u][0] = l < nb ? p[l] : 0.0;
            f[u][1] = 64 + l < nb ? p[64 + l] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int r = r0 + u * TRI_W;
            if (r >= nb)
                continue;
            if (l < nb)
                lds[ut ? r * R + l : l * R + r] = f[u][0];
            if (64 + l < nb)
                lds[ut ? r * R + 64 + l : (64 + l) * R + r] = f[u][1];
        }
    }
    __syncthreads();
    const int i0 = l < nb ? l : 0, i1 = 64 + l < nb ? 64 + l : 0;
    const double d0 = 1.0 / lds[i0 * R + i0], d1 = 1.0 / lds[i1 * R + i1];
    auto T = [&](int q) { return (const double *)(lds + q * R); };
    for (int v = first + w; v < s.count; v += step) {
        const double *p = s.in + v * s.vs;
        double y0 = p[i0 * s.es], y1 = p[i1 * s.es];
        if (ut)
            tri_forward<false>(nb, T, d0, d1, y0, y1);
        else if (s.kind & TRI_FORWARD)
            tri_forward<true>(nb, T, d0, d1, y0, y1);
        if (s.kind & TRI_BACKWARD)
            tri_backward(nb, T, y0, y1);
        double *o = s.out + v * s.vs;
        if (l < nb)
            o[i0 * s.es] = y0;
        if (64 + l < nb)
            o[i1 * s.es] = y1;
    }
}

// workgroups of a set: TRI_W vectors each
__host__ __device__ inline int tri_groups(int count) { return (count + TRI_W - 1) / TRI_W; }

__global__ __launch_bounds__(TRI_W * 64) void lu_tri_kernel(int nb, const double *F, long ldf,
                                                            TriSet s0, TriSet s1, TriSet s2)
{
    extern __shared__ double lds[];
    int g = blockIdx.x;
    if (g < tri_groups(s0.count)) {
        tri_body(nb, F, ldf, s0, g * TRI_W, s0.count, lds);
    } else if ((g -= tri_groups(s0.count)) < tri_groups(s1.count)) {
        tri_body(nb, F, ldf, s1, g * TRI_W, s1.count, lds);
    } else {
        g -= tri_groups(s1.count);
        tri_body(nb, F, ldf, s2, g * TRI_W, s2.count, lds);
    }
}

// ---- block products ---------------------------------------------------------------

// out = in - A B for an M x K block, A M x nb and B nb x K, nb <= 128: each
// element subtracts its products one after the other, q ascending (or, `desc`,
// descending), rounded separately.  A workgroup takes 32 x 32 elements, 2 x 2 a
// lane, its 32 rows of A and 32 columns of B in LDS.
struct MulSet {
    const double *A, *B, *in;
    double *out;
    long lda, ldb, ldi, ldo;
    int M, K;
};

__global__ __launch_bounds__(256) void lu_mul_kernel(int nb, MulSet s0, MulSet s1, int g0,
                                                     int desc)
{
    __shared__ double sa[LU_B][33], sb[LU_B][33];
    const MulSet &s = (int)blockIdx.x < g0 ? s0 : s1;
    const int g = (int)blockIdx.x < g0 ? blockIdx.x : blockIdx.x - g0;
    const int gk = (s.K + 31) / 32;
    const int r0 = g / gk * 32, c0 = g % gk * 32;
    const int t = threadIdx.x;
    for (int e = t; e < 32 * nb; e += 256) {
        const int r = e / nb, q = e % nb;
        sa[q][r] = r0 + r < s.M ? s.A[(long)(r0 + r) * s.lda + q] : 0.0;
    }
    for (int e = t; e < 32 * nb; e += 256) {
        const int q = e / 32, c = e % 32;
        sb[q][c] = c0 + c < s.K ? s.B[(long)q * s.ldb + c0 + c] : 0.0;
    }
    const int tr = t / 16, tc = t % 16;
    double v[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int r = r0 + tr + 16 * i, c = c0 + tc + 16 * j;
            v[i][j] = r < s.M && c < s.K ? s.in[(long)r * s.ldi + c] : 0.0;
        }
    __syncthreads();
#pragma unroll 4
    for (int e = 0; e < nb; e++) {
        const int q = desc ? nb - 1 - e : e;
        const double a0 = sa[q][tr], a1 = sa[q][tr + 16], b0 = sb[q][tc], b1 = sb[q][tc + 16];
        v[0][0] = sub_rn(v[0][0], mul_rn(a0, b0));
        v[0][1] = sub_rn(v[0][1], mul_rn(a0, b1));
        v[1][0] = sub_rn(v[1][0], mul_rn(a1, b0));
        v[1][1] = sub_rn(v[1][1], mul_rn(a1, b1));
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int r = r0 + tr + 16 * i, c = c0 + tc + 16 * j;
            if (r < s.M && c < s.K)
                s.out[(long)r * s.ldo + c] = v[i][j];
        }
}

__global__ __launch_bounds__(256) void lu_copy_kernel(long count, const double *__restrict__ src,
                                                      double *__restrict__ dst)
{
    for (long e = (long)blockIdx.x * 256 + threadIdx.x; e < count; e += (long)gridDim.x * 256)
        dst[e] = src[e];
}

// ---- the reference's backward substitution ------------------------------------------

// x_i = y_i - sum of x_q u_iq, q = i + 1, i + 2, ... subtracted in that order: row
// i can only start once x_{i+1} is known, so a column is one chain of
// N (N - 1) / 2 dependent subtractions.  One wave per workgroup, a lane per
// column (cw of them); the columns lie in LDS, entry q of lane c at c S + q with S
// even and S / 2 odd, so two entries come with one 16-byte read; u_iq is the same
// for all lanes (scalar loads).  In place on x.
__global__ __launch_bounds__(64) void lu_back_ref_kernel(int N, const double *__restrict__ gw,
                                                         int k, double *__restrict__ x, int cw)
{
    extern __shared__ double xs[];
    const int S = (N + 1) / 2 * 2 + ((N + 1) / 2 % 2 == 0 ? 2 : 0);
    const int c0 = blockIdx.x * cw, t = threadIdx.x;
    const int kw = k - c0 < cw ? k - c0 : cw;
    for (long e = t; e < (long)N * kw; e += 64)
        xs[e % kw * S + e / kw] = x[e / kw * k + c0 + e % kw];
    __syncthreads();
    const int c = t < kw ? t : 0;
    double *col = xs + (long)c * S;
    for (int i = N - 2; i >= 0; i--) {
        const double *u = gw + (long)i * N;
        double xi = col[i];
        int q = i + 1;
        if (q & 1) {
            xi = sub_rn(xi, mul_rn(col[q], u[q]));
            q++;
        }
        for (; q + 16 <= N; q += 16) {
            double2 w[8];
#pragma unroll
            for (int e = 0; e < 8; e++)
                w[e] = *(const double2 *)(col + q + 2 * e);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                xi = sub_rn(xi, mul_rn(w[e].x, u[q + 2 * e]));
                xi = sub_rn(xi, mul_rn(w[e].y, u[q + 2 * e + 1]));
            }
        }
        for (; q < N; q++)
            xi = sub_rn(xi, mul_rn(col[q], u[q]));
        if (t < kw)
            col[i] = xi;
    }
    __syncthreads();
    for (long e = t; e < (long)N * kw; e += 64)
        x[e / kw * k + c0 + e % kw] = xs[e % kw * S + e / kw];
}

// The same for N <= 128, four columns to a wave: lane l holds entries l % 16, 16 +
// l % 16, ... of column l / 16.  The products of 16 entries with a row of U are one
// instruction, and sixteen v_fmac_f64 (x -1) take them in turn by DPP
// (row_newbcast), each a subtraction rounded once, so a step of the chain costs the
// wave one FP64 issue (8.5 cycles) instead of a product, a subtraction and their
// operand reads.  U lies in LDS, its next row read while the current one runs.
// Entries at or before i give zero products, which change nothing.
// N = 128, the substitution alone: k = 16 164 -> about 30 us, k = 128 304 -> 32 us.
constexpr int LB_W = 4;   // waves (of 4 columns) of a workgroup

__device__ __forceinline__ void chain16_sub(double &acc, double v)
{
    const double minus = -1.0;
    // s_nop: a DPP read comes two wait states after the write of its register
#define CACG_LB(r) "v_fmac_f64_dpp %0, %1, %2 row_newbcast:" #r " row_mask:0xf bank_mask:0xf\n\t"
    asm("s_nop 1\n\t" CACG_LB(0) CACG_LB(1) CACG_LB(2) CACG_LB(3) CACG_LB(4) CACG_LB(5) CACG_LB(6)
            CACG_LB(7) CACG_LB(8) CACG_LB(9) CACG_LB(10) CACG_LB(11) CACG_LB(12) CACG_LB(13)
                CACG_LB(14) CACG_LB(15)
        : "+&v"(acc)
        : "v"(v), "v"(minus));
#undef CACG_LB
}

// rows 16 B + 15 .. 16 B of one column block, then the blocks before it; NB blocks
// of 16 rows in all
template <int NB, int B>
__device__ __forceinline__ void back_block(double (&x)[NB], const double *us, const double *yc,
                                           int S, int lane)
{
    double u[NB - B];
    auto read = [&](double *w, int i) {
#pragma unroll
        for (int b = B; b < NB; b++)
            w[b - B] = us[i * S + 16 * b + lane];
    };
    read(u, 16 * B + 15);
    double y = yc[16 * B + 15];
    for (int il = 15; il >= 0; il--) {
        const int i = 16 * B + il, in = il > 0 ? i - 1 : i;
        double un[NB - B];
        read(un, in);
        const double yn = yc[in];
        double p[NB - B];
#pragma unroll
        for (int b = NB - 1; b > B; b--)
            p[b - B] = mul_rn(x[b], u[b - B]);
        p[0] = lane > il ? mul_rn(x[B], u[0]) : 0.0;
        double acc = y;
#pragma unroll
        for (int b = B; b < NB; b++)
            chain16_sub(acc, p[b - B]);
        x[B] = lane == il ? acc : x[B];
#pragma unroll
        for (int b = 0; b < NB - B; b++)
            u[b] = un[b];
        y = yn;
    }
    if constexpr (B > 0)
        back_block<NB, B - 1>(x, us, yc, S, lane);
}

// dynamic LDS: U (16 NB x 16 NB, zeros past N), then y of each column
template <int NB>
__global__ __launch_bounds__(LB_W * 64) void lu_back16_ref_kernel(int N,
                                                                  const double *__restrict__ gw,
                                                                  int k, double *__restrict__ x)
{
    extern __shared__ double us[];
    constexpr int R = 16 * NB, S = R;
    double *ys = us + R * S;   // entry i of column c at ys + c (R + 1) + i
    const int t = threadIdx.x, c0 = blockIdx.x * LB_W * 4;
    for (int e = t; e < R * R; e += LB_W * 64) {
        const int i = e / R, q = e % R;
        us[i * S + q] = i < N && q < N ? gw[(long)i * N + q] : 0.0;
    }
    for (int e = t; e < R * LB_W * 4; e += LB_W * 64) {
        const int i = e / (LB_W * 4), c = e % (LB_W * 4);
        ys[c * (R + 1) + i] = i < N && c0 + c < k ? x[(long)i * k + c0 + c] : 0.0;
    }
    __syncthreads();
    const int lane = t & 15, c = t >> 4;
    double v[NB];
#pragma unroll
    for (int b = 0; b < NB; b++)
        v[b] = 0.0;
    back_block<NB, NB - 1>(v, us, ys + c * (R + 1), S, lane);
    __syncthreads();
#pragma unroll
    for (int b = 0; b < NB; b++)
        ys[c * (R + 1) + 16 * b + lane] = v[b];
    __syncthreads();
    for (int e = t; e < N * LB_W * 4; e += LB_W * 64) {
        const int i = e / (LB_W * 4), cc = e % (LB_W * 4);
        if (c0 + cc < k)
            x[(long)i * k + c0 + cc] = ys[cc * (R + 1) + i];
    }
}

template <int NB>
int launch_back16(int N, const double *gw, int k, double *x, hipStream_t st)
{
    constexpr int R = 16 * NB;
    const size_t shm = ((size_t)R * R + LB_W * 4 * (R + 1)) * sizeof(double);
    cacg_allow_lds(lu_back16_ref_kernel<NB>, shm);
    hipLaunchKernelGGL(lu_back16_ref_kernel<NB>, dim3((k + LB_W * 4 - 1) / (LB_W * 4)),
                       dim3(LB_W * 64), shm, st, N, gw, k, x);
    CACG_LAUNCH_CHECK();
    return 0;
}

// ---- batched ------------------------------------------------------------------------

// workgroup b factors system items[b].x (N = sm <= 128, m <= 32): alpha = QtAQ^{-1} QtR
__global__ __launch_bounds__(LU_T) void lu_batch_alpha_kernel(const cacg_bsys *__restrict__ sys,
                                                              const int2 *__restrict__ items)
{
    extern __shared__ double lds[];
    const cacg_bsys &d = sys[items[blockIdx.x].x];
    lu_factor_body(d.sm, d.QtAQ, d.sm, d.lu, d.sm, d.m, d.QtR, d.alpha, d.flag, true, lds);
}

// beta = QtAQ^{-1} QtAS with the factor kept from the last alpha solve; workgroup
// (b, y) takes columns TRI_W y .., in steps of TRI_W gridDim.y
__global__ __launch_bounds__(TRI_W * 64) void lu_batch_beta_kernel(
    const cacg_bsys *__restrict__ sys, const int2 *__restrict__ items)
{
    extern __shared__ double lds[];
    const cacg_bsys &d = sys[items[blockIdx.x].x];
    if ((int)blockIdx.y * TRI_W >= d.sm)
        return;
    const TriSet s = {d.QtAS, d.beta, 1, d.sm, d.sm, TRI_FORWARD | TRI_BACKWARD};
    tri_body(d.sm, d.lu, d.sm, s, blockIdx.y * TRI_W, TRI_W * gridDim.y, lds);
}

int launch_factor(int N, const double *lhs, long ldl, double *gw, long ldg, int k,
                  const double *rhs, double *x, int *flag, int back, hipStream_t st)
{
    const size_t shm = (size_t)lu_factor_lds(N, k, back != 0) * sizeof(double);
    cacg_allow_lds(lu_factor_kernel, shm);
    hipLaunchKernelGGL(lu_factor_kernel, dim3(1), dim3(LU_T), shm, st, N, lhs, ldl, gw, ldg, k,
                       rhs, x, flag, back);
    CACG_LAUNCH_CHECK();
    return 0;
}

const TriSet TRI_NONE = {nullptr, nullptr, 0, 0, 0, 0};

int launch_tri(int nb, const double *F, long ldf, const TriSet &a, const TriSet &b,
               const TriSet &c, hipStream_t st)
{
    const int G = tri_groups(a.count) + tri_groups(b.count) + tri_groups(c.count);
    if (G == 0)
        return 0;
    const size_t shm = (size_t)tri_lds(nb) * sizeof(double);
    cacg_allow_lds(lu_tri_kernel, shm);
    hipLaunchKernelGGL(lu_tri_kernel, dim3(G), dim3(TRI_W * 64), shm, st, nb, F, ldf, a, b, c);
    CACG_LAUNCH_CHECK();
    return 0;
}

int launch_mul(int nb, const MulSet &a, const MulSet &b, int desc, hipStream_t st)
{
    const int ga = (a.M + 31) / 32 * ((a.K + 31) / 32), gb = (b.M + 31) / 32 * ((b.K + 31) / 32);
    if (ga + gb == 0)
        return 0;
    hipLaunchKernelGGL(lu_mul_kernel, dim3(ga + gb), dim3(256), 0, st, nb, a, b, ga, desc);
    CACG_LAUNCH_CHECK();
    return 0;
}

#define LU_TRY(call)                                                                              \
    do {                                                                                          \
        const int rc_ = (call);                                                                   \
        if (rc_)                                                                                  \
            return rc_;                                                                           \
    } while (0)

// N > 128 in blocks of 128.  Right-looking, so each element receives its
// subtractions in ascending order of the pivot, block after block.  `factor`:
// factor first, the right-hand sides (fewer columns of the same steps) along
// with it; else the factor is in gw.  In x afterwards: y = L^{-1} rhs for a
// reference-order backward pass (`back` false), or x.
int lu_blocked(int N, int k, const double *rhs, double *x, double *gw, int *flag, bool factor,
               bool back, hipStream_t st)
{
    for (int p = 0; p < N; p += LU_B) {
        const int nb = N - p < LU_B ? N - p : LU_B, rest = N - p - nb, e = p + nb;
        double *F = gw + (long)p * N + p;
        // the first block's right-hand side rows come from rhs, later ones have
        // been updated into x
        const double *in = p == 0 ? rhs : x + (long)p * k;
        double *xp = x + (long)p * k;
        // the last block's backward pass follows its forward pass
        const int kind = TRI_FORWARD | (back && rest == 0 ? TRI_BACKWARD : 0);
        if (factor)
            LU_TRY(launch_factor(nb, F, N, F, N, 0, nullptr, nullptr, flag, 0, st));
        const TriSet y = {in, xp, 1, k, k, kind};
        const TriSet u = {gw + (long)p * N + e, gw + (long)p * N + e, 1, N, rest, TRI_FORWARD};
        const TriSet l = {gw + (long)e * N + p, gw + (long)e * N + p, N, 1, rest, TRI_UT};
        LU_TRY(launch_tri(nb, F, N, y, factor ? u : TRI_NONE, factor ? l : TRI_NONE, st));
        if (rest == 0)
            break;
        double *L = gw + (long)e * N + p, *A = gw + (long)e * N + e;
        const double *rin = p == 0 ? rhs + (long)e * k : x + (long)e * k;
        const MulSet ry = {L, xp, rin, x + (long)e * k, N, k, k, k, rest, k};
        MulSet ra = {L, gw + (long)p * N + e, A, A, N, N, N, N, rest, rest};
        if (!factor)
            ra.M = ra.K = 0;
        LU_TRY(launch_mul(nb, ry, ra, 0, st));
    }
    if (!back)
        return 0;
    for (int p = (N - 1) / LU_B * LU_B; p > 0; p -= LU_B) {
        // x above block p subtracts U(:, block) x(block), then the block above it
        const int nb = N - p < LU_B ? N - p : LU_B;
        const MulSet up = {gw + p, x + (long)p * k, x, x, N, k, k, k, p, k};
        LU_TRY(launch_mul(nb, up, MulSet{}, 1, st));
        const int q = p - LU_B;
        const TriSet b = {x + (long)q * k, x + (long)q * k, 1, k, k, TRI_BACKWARD};
        LU_TRY(launch_tri(LU_B, gw + (long)q * N + q, N, b, TRI_NONE, TRI_NONE, st));
    }
    return 0;
}

}  // namespace

extern "C" int cacg_k_lu_batch(const cacg_bsys *d_sys, const int2 *d_items, int count, int which,
                               int max_sm, hipStream_t st)
{
    if (count <= 0)
        return 0;
    if (max_sm <= 0 || max_sm > 128 || (which != 0 && which != 1))
        return (int)hipErrorInvalidValue;
    if (which == 1) {
        const size_t shm = (size_t)lu_factor_lds(max_sm, LU_K, true) * sizeof(double);
        cacg_allow_lds(lu_batch_alpha_kernel, shm);
        hipLaunchKernelGGL(lu_batch_alpha_kernel, dim3(count), dim3(LU_T), shm, st, d_sys,
                           d_items);
    } else {
        const size_t shm = (size_t)tri_lds(max_sm) * sizeof(double);
        cacg_allow_lds(lu_batch_beta_kernel, shm);
        hipLaunchKernelGGL(lu_batch_beta_kernel, dim3(count, (max_sm + 15) / 16),
                           dim3(TRI_W * 64), shm, st, d_sys, d_items);
    }
    CACG_LAUNCH_CHECK();
    return 0;
}

extern "C" int cacg_k_lu_solve(int N, const double *lhs, int k, const double *rhs, double *x,
                               double *d_work, int *d_flag, int mode, int reuse_factor,
                               hipStream_t st)
{
    if (N <= 0 || k <= 0 || N > 16384)
        return (int)hipErrorInvalidValue;
    const bool fast = mode == CACG_MODE_FAST;
    const bool factor = !reuse_factor;
    if (N <= LU_B) {
        const bool along = factor && k <= LU_K;   // the right-hand sides with the factorisation
        if (factor)
            LU_TRY(launch_factor(N, lhs, N, d_work, N, along ? k : 0, rhs, x, d_flag,
                                 along && fast, st));
        if (!along) {
            const TriSet s = {rhs, x, 1, k, k, TRI_FORWARD | (fast ? TRI_BACKWARD : 0)};
            LU_TRY(launch_tri(N, d_work, N, s, TRI_NONE, TRI_NONE, st));
        }
    } else {
        if (factor) {
            hipLaunchKernelGGL(lu_copy_kernel, dim3(cacg_grid((long)N * N, 256, 1024)), dim3(256),
                               0, st, (long)N * N, lhs, d_work);
            CACG_LAUNCH_CHECK();
        }
        LU_TRY(lu_blocked(N, k, rhs, x, d_work, d_flag, factor, fast, st));
    }
    if (!fast && N <= 128) {
        switch ((N + 15) / 16) {
        case 1: return launch_back16<1>(N, d_work, k, x, st);
        case 2: return launch_back16<2>(N, d_work, k, x, st);
        case 3: return launch_back16<3>(N, d_work, k, x, st);
        case 4: return launch_back16<4>(N, d_work, k, x, st);
        case 5: return launch_back16<5>(N, d_work, k, x, st);
        case 6: return launch_back16<6>(N, d_work, k, x, st);
        case 7: return launch_back16<7>(N, d_work, k, x, st);
        default: return launch_back16<8>(N, d_work, k, x, st);
        }
    }
    if (!fast) {
        // columns per workgroup: 16, fewer where N x 16 doubles exceed 128 KiB
        const int S = N + 3;
        int cw = 16384 / S;
        cw = cw > 16 ? 16 : cw < 1 ? 1 : cw;
        const size_t shm = (size_t)cw * S * sizeof(double);
        cacg_allow_lds(lu_back_ref_kernel, shm);
        hipLaunchKernelGGL(lu_back_ref_kernel, dim3((k + cw - 1) / cw), dim3(64), shm, st, N,
                           d_work, k, x, cw);
        CACG_LAUNCH_CHECK();
    }
    return 0;
}
