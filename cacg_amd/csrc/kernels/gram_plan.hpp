// Plans of the fast-order Gram and the loads of its tile kernel: which rows a
// workgroup takes, which tiles its waves form, and which vectors of a stage each lane
// loads.  Nothing here needs a GPU, so the bounds of every load can be walked on the
// host with the same code that the kernel runs.
#pragma once

#include <stddef.h>

#include <initializer_list>

#ifdef __HIPCC__
#include <hip/hip_runtime.h>

#define CACG_HD __host__ __device__ __forceinline__
#else
#define CACG_HD inline
#endif

struct GramPlan {
    int TM, TN;   // 16x16 tiles in M (kl) and N (kr)
    int KS;       // 1 from four groups of tiles on (see plan_gram), else more
    int gx;       // row chunks (split K across workgroups)
    int chunk;    // rows per chunk
};

// The chunks, and with them the order of the sums, are a function of n and the widths
// only, not of the device: about 512 of them (2 workgroups a CU), fewer where a G is cut
// into many groups of 2 x 9 (or 1 x 9) tiles, at least 64 rows each.
inline GramPlan plan_gram(int n, int kl, int kr)
{
    GramPlan p;
    p.TM = (kl + 15) / 16;
    p.TN = (kr + 15) / 16;
    const int NT = p.TN < 9 ? p.TN : 9, MT = p.TM >= 8 ? 2 : 1;
    const int NG = (p.TM + MT - 1) / MT * ((p.TN + NT - 1) / NT);
    p.KS = NG >= 4 ? 1 : 4 / NG;
    int gx = 512 / ((NG + 3) / 4);
    if (gx < 1)
        gx = 1;
    // whole stages of the 128-column kernels (16 rows), else of 8 rows a share
    const int step = p.TM == 8 ? 16 : 8 * p.KS;
    const long maxc = ((long)n + 63) / 64;
    if (gx > maxc)
        gx = (int)(maxc > 0 ? maxc : 1);
    long chunk = ((long)n + gx - 1) / gx;
    chunk = (chunk + step - 1) / step * step;
    if (chunk < step)
        chunk = step;
    p.chunk = (int)chunk;
    p.gx = (int)(((long)n + chunk - 1) / chunk);
    if (p.gx < 1)
        p.gx = 1;
    return p;
}

// LDS row stride (doubles) of a staged k-column block: k rounded up to 16
// mod 32.  A wave reads 4 rows x 16 consecutive doubles per MFMA operand;
// with a stride of 16 mod 32 doubles, rows 0, 1 (and 2, 3) fall into the two
// disjoint halves of the 64 four-byte LDS banks, so a 64-lane read takes the
// 2 cycles its 512 bytes need (a stride of k + 2 overlapped all four rows).
CACG_HD int lds_row_stride(int k)
{
    return k + (48 - k % 32) % 32;
}

// ---- the tile kernel ----------------------------------------------------------------

struct GramTile {
    int TMB, TNB;    // tiles of a block
    int nbn;         // blocks along N
    int GN, NG, KS;  // groups along N, groups, row shares
    int MT, NT, VEC;
    int W;           // waves the kernel is built for: 16, or 8 with twice the registers
    size_t lds;
};

constexpr int GT_TM = 8, GT_TN = 10;

// loads of a stage per lane
CACG_HD constexpr int gt_loads(int W, int VEC)
{
    return W == 16 ? (VEC == 2 ? 3 : 5) : (VEC == 2 ? 5 : 9);
}

// at least 128 rows a chunk, half the partials: from 8192 rows on where a block's few
// tiles leave waves for more row shares (4 + 4 columns against 4, 20,000 rows: 14.0 -> 11.3
// us; 100 columns: 28 -> 31 us, not taken), and from 3072 to 8192 rows where a partial is
// large (256 + 32 columns, 5000 rows: 46.5 -> 36.9 us; 10,000: 60 -> 64, not taken)
inline void tile_chunks(int n, GramPlan &p)
{
    const int tiles = p.TM * p.TN;
    if (p.chunk < 128 && (n >= 8192 ? tiles <= 24 : n >= 3072 && tiles >= 100)) {
        p.chunk = 128;
        p.gx = (n + 127) / 128;
    }
}

// the tile group and row shares of a block: the fewest MFMA slots per row on the
// busiest SIMD (waves are dealt round-robin over 4), then the most waves; at
// most 16 waves and 80 KiB of LDS (two workgroups a CU) while a single row share
// allows it
//
// gx: row chunks.  With fewer workgroups than half the CUs the blocks are halved, the
// longer side first, until there are: the chip is idle then, and a chunk's tiles take
// the longer the more of them one CU forms (2000 rows, 112 + 16 columns: 19.4 ->
// 10.8 us; 256 or 512 workgroups instead of 128: 14 to 16).
// f32: R1 is FP32 and its vectors start at a wave's first lane.
inline GramTile plan_tile(int TM, int TN, int VEC, int chunk, int gx, bool f32)
{
    static const int shape[][2] = {{1, 1}, {1, 2}, {1, 3}, {1, 4}, {1, 5}, {2, 2}, {2, 3}};
    GramTile best{};
    int bm = (TM + GT_TM - 1) / GT_TM, bn = (TN + GT_TN - 1) / GT_TN;
    while (gx * bm * bn <= 128 && (bm < TM || bn < TN)) {
        if ((TM + bm - 1) / bm >= (TN + bn - 1) / bn)
            bm = 2 * bm < TM ? 2 * bm : TM;
        else
            bn = 2 * bn < TN ? 2 * bn : TN;
    }
    best.TMB = (TM + bm - 1) / bm;
    best.TNB = (TN + bn - 1) / bn;
    best.nbn = (TN + best.TNB - 1) / best.TNB;
    best.VEC = VEC;
    double cost = 1e30;
    const int cols = lds_row_stride(best.TMB * 16) + lds_row_stride(best.TNB * 16);
    for (const auto &sh : shape) {
        const int MT = sh[0], NT = sh[1];
        const int GM = (best.TMB + MT - 1) / MT, GN = (best.TNB + NT - 1) / NT, NG = GM * GN;
        // no more row shares than 16-row pieces in a chunk
        for (int KS = 1; NG * KS <= 16 && (KS == 1 || 16 * KS <= chunk); KS++) {
            const int W = NG * KS <= 8 ? 8 : 16;
            // loads of a row: L, R1 and R2 may each end with an odd column
            const int row = 16 * (best.TMB + best.TNB) / VEC + VEC - 1;
            if (16 * KS * row + (f32 ? 63 : 0) > 64 * gt_loads(W, VEC) * NG * KS)
                continue;
            const size_t stage = 2 * (size_t)(16 * KS * cols + 32) * sizeof(double);
            const size_t red = (size_t)(KS - 1) * NG * MT * NT * 256 * sizeof(double);
            const size_t lds = stage > red ? stage : red;
            if (lds > (KS == 1 ? 160 : 80) * 1024)
                break;
            const double c = (double)((NG * KS + 3) / 4) * MT * NT / KS - 1e-3 * NG * KS;
            if (c < cost) {
                cost = c;
                best.GN = GN;
                best.NG = NG;
                best.KS = KS;
                best.MT = MT;
                best.NT = NT;
                best.W = W;
                best.lds = lds;
            }
        }
    }
    return best;
}

// whether every source has two columns in every block it reaches, R2 possibly one
// column in all: a block that holds a single one of a wider source cannot pair it
inline bool tile_pairs(int n, int kl, int kr1, int kr2, const GramTile &g)
{
    auto lone = [](int w, int k) { return k > 0 && k % w == 1; };
    const int w = g.TNB * 16, e1 = kr1 % w;   // columns of R1 before R2 in their block
    const int first2 = kr2 < w - e1 ? kr2 : w - e1;
    const bool r2 = kr2 > 1 && (first2 == 1 || lone(w, kr2 - first2));
    return !(n < 2 || lone(g.TMB * 16, kl) || lone(w, kr1) || r2);
}

// the plan with two columns a load, with the blocks halved for idle CUs or, where that
// leaves a single column to a block, without; false: single columns
inline bool plan_pairs(int n, int kl, int kr1, int kr2, const GramPlan &p, bool f32, GramTile &g)
{
    for (int gx : {p.gx, 129}) {
        g = plan_tile(p.TM, p.TN, 2, p.chunk, gx, f32);
        // a single column of R2 has a load of its own, in FP64 blocks of one or two tiles a wave
        const bool one = kr2 == 1 && (f32 || g.MT * g.NT > 2);
        if (g.NG && !one && tile_pairs(n, kl, kr1, kr2, g))
            return true;
    }
    return false;
}

// The vectors of a stage of SR rows: VEC columns each, L's row by row, then those of
// [R1 | R2] row by row, without R2's where it is a single column (ONE).  A last odd
// column's pair starts one column early, inside the row.  F32: R1 is FP32, and the
// second part starts at a wave's first lane, so that no wave loads both types (it would
// do so one after the other, and all waves wait for it at the stage's end: 2,097,152
// rows of 60 columns 705 -> 517 us).
template <int VEC, bool ONE, bool F32>
struct GtStage {
    int SR, kl, k1, k2;   // columns of the block: L's, R1's, R2's
    int wl, w1, wr;       // vectors of a row of L, of R1, of [R1 | R2]
    int second;           // first vector of [R1 | R2]
    int LDP, RDP;
    float il, ir;
    CACG_HD GtStage(int SR_, int kl_, int k1_, int k2_)
        : SR(SR_), kl(kl_), k1(k1_), k2(k2_), wl((kl_ + VEC - 1) / VEC), w1((k1_ + VEC - 1) / VEC),
          wr((k1_ + VEC - 1) / VEC + (ONE ? 0 : (k2_ + VEC - 1) / VEC)),
          second(F32 ? (SR_ * wl + 63) / 64 * 64 : SR_ * wl), LDP(lds_row_stride(kl_)),
          RDP(lds_row_stride(k1_ + k2_)), il(1.0f / wl), ir(1.0f / wr)
    {
    }
    CACG_HD int count() const { return second + SR * wr; }
    CACG_HD static int start(int q, int k) { return VEC * q + VEC <= k || VEC == 1 ? VEC * q : k - VEC; }
    // vector v's LDS offset, source (0 L, 1 R1, 2 R2) and row, packed; ~0u past the
    // last; col: its first column in L's or in [R1 | R2]'s part of the block.  The
    // divisions: v / w for v < 2^14, w <= 256 (the error of the product is far below
    // 0.5 / w).
    CACG_HD unsigned vector(int v, int &col) const
    {
        col = 0;
        if (v < SR * wl) {
            const int row = (int)((v + 0.5f) * il);
            col = start(v - row * wl, kl);
            return (unsigned)(row * LDP + col) << 12 | row;
        }
        if ((v -= second) >= 0 && v < SR * wr) {
            const int row = (int)((v + 0.5f) * ir), q = v - row * wr;
            col = q < w1 ? start(q, k1) : k1 + start(q - w1, k2);
            return (unsigned)(SR * LDP + row * RDP + col) << 12 | (q < w1 ? 1u : 2u) << 10 | row;
        }
        return ~0u;
    }
};

CACG_HD int gt_row(unsigned info) { return info & 1023; }
CACG_HD int gt_kind(unsigned info) { return info >> 10 & 3; }

// rows of a stage that a chunk of `rows` rows has; a lane loads its vector if its row
// is among them.  At most SR <= 256, so that a lane without a vector (row 1023) loads
// nothing however many rows the chunk still has.
CACG_HD int gt_stage_rows(int rows, int SR, int st)
{
    const int left = rows - st * SR;
    return left < SR ? left : SR;
}
