// Tall-skinny QR of an n x k block (k <= 128): A = Q R, Q n x k with
// orthonormal columns, R k x k upper triangular with a positive diagonal.
// gfx950.
//
// Algorithm: CholeskyQR2.  One pass is G = A^T A (the split-K FP64 MFMA
// Gram, a deterministic fixed-order reduction), R1 = chol(G) and
// W = R1^{-1} in one workgroup, then Q1 = A W (the tall-skinny
// MFMA update); the second pass repeats it on Q1 and R = R2 R1.  The second
// pass brings the loss of orthogonality from O(u cond(A)^2) down to O(u) for
// cond(A) up to about u^{-1/2} (1e8); a Cholesky pivot that is not finite or
// not above 64 u times its original diagonal entry (A numerically rank
// deficient, or cond(A) beyond that range) sets *d_flag.
// No reference counterpart: the reference's TSQR.c is empty.
#include <math.h>

#include <type_traits>

#include "kcommon.hpp"

namespace {

constexpr int QT = 1024;
constexpr int QP = 8;      // pivots of a panel
constexpr int QS = 10;     // LDS stride of a panel column (16-byte reads, all 64 banks)

// G (N x N, row-major, symmetric positive definite, N <= 128) -> R (upper, the
// lower triangle written as zeros) and W = -R^{-1} (upper, zeros below).
//
// Right-looking Cholesky of the upper triangle with the identity as further
// columns: the elimination that turns G into R turns the identity into
// Y = R^{-T}, so the inverse costs no pass of its own.  Lane (tr, tc) of a
// 32 x 32 grid keeps elements (tr + 32 i, tc + 32 j) in registers, of G for
// i <= j and of Y for i >= j.  Per panel of 8 rows: three waves, a column a lane,
// factor it, each with the diagonal block's 8 columns beside its own 56 (rows
// are passed by readlane, no barrier inside the panel); then every lane applies
// the 8 updates to its elements and the owners of the next panel put it into
// LDS.  Bound by the chain of pivots (square root, reciprocal, product, update).
// Before, with three barriers and a pass over LDS for every pivot and one lane a
// column of the inverse: 562 us at N = 96.
__global__ __launch_bounds__(QT) void chol_inv_kernel(int N, const double *__restrict__ G,
                                                      double *__restrict__ R,
                                                      double *__restrict__ W, int *flag)
{
    __shared__ double rp[128 * QS], yp[128 * QS], g0[128];
    const int t = threadIdx.x, tr = t >> 5, tc = t & 31;
    const int wave = t >> 6, lane = t & 63;
    double v[4][4], y[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int r = tr + 32 * i, c = tc + 32 * j;
            const bool in = r < N && c < N;
            if (i <= j)
                v[i][j] = in ? G[r * N + c] : (r == c ? 1.0 : 0.0);
            if (i >= j)
                y[i][j] = r == c ? 1.0 : 0.0;
            if (in && r > c) {
                R[r * N + c] = 0.0;
                W[r * N + c] = 0.0;
            }
        }
    for (int e = t; e < 128 * QS; e += QT)
        yp[e] = 0.0;
    if (t < 128)
        g0[t] = t < N ? G[t * N + t] : 1.0;
    __syncthreads();
    auto publish = [&](auto I, int q0) {
        constexpr int ip = decltype(I)::value;
        const int dr = tr - q0;
        if (dr >= 0 && dr < QP) {
#pragma unroll
            for (int j = ip; j < 4; j++)
                rp[(tc + 32 * j) * QS + dr] = v[ip][j];
#pragma unroll
            for (int j = 0; j <= ip; j++)
                yp[(tc + 32 * j) * QS + dr] = y[ip][j];
        }
    };
    // rows above the next panel are final and stored; they take part unread
    auto update = [&](auto I) {
        constexpr int ip = decltype(I)::value;
#pragma unroll 1
        for (int p = 0; p < QP; p += 2) {
            double2 l[4];
#pragma unroll
            for (int i = ip; i < 4; i++)
                l[i] = *(const double2 *)(rp + (tr + 32 * i) * QS + p);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const double2 w = *(const double2 *)(yp + (tc + 32 * j) * QS + p);
#pragma unroll
                for (int i = ip > j ? ip : j; i < 4; i++)
                    y[i][j] = y[i][j] - l[i].x * w.x - l[i].y * w.y;
            }
#pragma unroll
            for (int j = ip; j < 4; j++) {
                const double2 u = *(const double2 *)(rp + (tc + 32 * j) * QS + p);
#pragma unroll
                for (int i = ip; i <= j; i++)
                    v[i][j] = v[i][j] - l[i].x * u.x - l[i].y * u.y;
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
    for (int P0 = 0; P0 < N; P0 += QP) {
        const int P1 = P0 + QP;
        const int right = N - P1 > 0 ? N - P1 : 0;   // columns of G right of the panel
        const int left = P1 < N ? P1 : N;            // columns of Y that are not zero yet
        if (wave < (right + left + 55) / 56) {
            const int e = wave * 56 + lane - QP;
            const bool diag = lane < QP, isy = !diag && e >= right;
            const bool in = !diag && e < right + left;
            const int c = diag ? P0 + lane : in ? (isy ? e - right : P1 + e) : 0;
            const double *src = isy && in ? yp + c * QS : rp + c * QS;
            double w[QP];
#pragma unroll
            for (int i = 0; i < QP; i++)
                w[i] = src[i];
            int bad = 0;
#pragma unroll
            for (int p = 0; p < QP; p++) {
                const double piv = readlane_f64(w[p], p);
                // a pivot below 64 u of its original diagonal entry has lost every
                // significant digit: its column is (numerically) in the span of the
                // ones before
                if (P0 + p < N && (!(piv > 0x1p-47 * g0[P0 + p]) || !isfinite(piv)))
                    bad = 1;
                const double d = sqrt(piv > 0.0 ? piv : 1.0);
                const double inv = 1.0 / d;
                w[p] = diag && lane == p ? d : w[p] * inv;
#pragma unroll
                for (int i = p + 1; i < QP; i++)
                    w[i] -= readlane_f64(w[p], i) * w[p];
            }
            if (in) {
#pragma unroll
                for (int i = 0; i < QP; i++) {
                    const int r = P0 + i;
                    if (isy)
                        yp[c * QS + i] = w[i];
                    else
                        rp[c * QS + i] = w[i];
                    if (r >= N)
                        continue;
                    if (!isy)
                        R[r * N + c] = w[i];
                    else if (c <= r)
                        W[c * N + r] = -w[i];
                }
            }
            if (wave == 0 && diag && c < N) {
#pragma unroll
                for (int i = 0; i < QP; i++)
                    if (i <= lane)
                        R[(P0 + i) * N + c] = w[i];
            }
            if (wave == 0 && lane == 0 && bad)
                *flag = 1;
        }
        __syncthreads();
        if (P1 >= N)
            break;
        switch (P0 / 32) {
        case 0: update(I0{}); break;
        case 1: update(I1{}); break;
        case 2: update(I2{}); break;
        default: update(I3{}); break;
        }
        __syncthreads();
        switch (P1 / 32) {
        case 0: publish(I0{}, P1 % 32); break;
        case 1: publish(I1{}, P1 % 32); break;
        case 2: publish(I2{}, P1 % 32); break;
        default: publish(I3{}, P1 % 32); break;
        }
        __syncthreads();
    }
}

// out = A B for upper triangular N x N A and B (N <= 128), zeros below; 16 x 16
// elements a workgroup
__global__ __launch_bounds__(256) void upper_mul_kernel(int N, const double *__restrict__ A,
                                                        const double *__restrict__ B,
                                                        double *__restrict__ out)
{
    __shared__ double sa[128][17], sb[128][17];
    const int t = threadIdx.x, tr = t / 16, tc = t % 16;
    const int r0 = blockIdx.y * 16, c0 = blockIdx.x * 16;
    if (c0 >= r0) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int j = tc + 16 * e, q = tr + 16 * e;
            sa[j][tr] = r0 + tr < N && j < N ? A[(r0 + tr) * N + j] : 0.0;
            sb[q][tc] = q < N && c0 + tc < N ? B[q * N + c0 + tc] : 0.0;
        }
    }
    __syncthreads();
    const int r = r0 + tr, c = c0 + tc;
    double s = 0.0;
    if (c0 >= r0) {
        const int e = c0 + 16 < N ? c0 + 16 : N;
#pragma unroll 4
        for (int j = r0; j < e; j++)
            s += sa[j][tr] * sb[j][tc];
    }
    if (r < N && c < N)
        out[r * N + c] = c >= r ? s : 0.0;
}

}  // namespace

extern "C" long cacg_tsqr_workspace(int k)
{
    // Gram partials, then G, R1, W, R2
    return cacg_gram_workspace(k, k) + 4L * k * k;
}

extern "C" int cacg_k_tsqr(int n, int k, const double *A, long lda, double *Q, double *R,
                           double *d_work, int *d_flag, hipStream_t st)
{
    if (n < 0 || k <= 0 || k > 128 || lda < k || !A || !Q || !R || !d_work || !d_flag)
        return (int)hipErrorInvalidValue;
    double *gw = d_work;
    double *G = gw + cacg_gram_workspace(k, k);
    double *R1 = G + (long)k * k, *W = R1 + (long)k * k, *R2 = W + (long)k * k;
    for (int pass = 0; pass < 2; pass++) {
        // the first pass reads A where it lies and writes Q, the second works on Q
        const double *in = pass == 0 ? A : Q;
        const long ld = pass == 0 ? lda : k;
        int rc = cacg_k_gram_fast(n, in, ld, k, in, ld, k, NULL, 0, 0, G, NULL, gw, st);
        if (rc)
            return rc;
        hipLaunchKernelGGL(chol_inv_kernel, dim3(1), dim3(QT), 0, st, k, G, pass == 0 ? R1 : R2,
                           W, d_flag);
        CACG_LAUNCH_CHECK();
        rc = cacg_k_trimul_neg(n, k, in, ld, Q, W, st);   // Q = in (-W)
        if (rc)
            return rc;
    }
    hipLaunchKernelGGL(upper_mul_kernel, dim3((k + 15) / 16, (k + 15) / 16), dim3(256), 0, st, k,
                       R2, R1, R);
    CACG_LAUNCH_CHECK();
    return 0;
}
