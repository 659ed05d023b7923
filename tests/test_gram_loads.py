"""Bounds of the loads of the fast-order Gram's tile kernel, walked on the host with the
plan and the lane mapping that the kernel itself is compiled from (gram_plan.hpp)."""

import os
import subprocess

import pytest

from conftest import ROOT

WALK = r"""
#include "gram_plan.hpp"

#include <cstdio>
#include <cstdlib>
#include <vector>

static void fail(const char *what, int a, int b, int c)
{
    std::printf("%s: %d %d %d\n", what, a, b, c);
    std::exit(1);
}

// every lane, load and stage kind of one block over rows r0 .. r1 - 1
template <int VEC, bool ONE, bool F32>
static void walk(const GramTile &g, int n, int kl_all, int kr1, int kr2, int r0, int r1, int by)
{
    const int ca = by / g.nbn * g.TMB * 16, cb = by % g.nbn * g.TNB * 16, krt = kr1 + kr2;
    const int kl = kl_all - ca < g.TMB * 16 ? kl_all - ca : g.TMB * 16;
    const int kr = krt - cb < g.TNB * 16 ? krt - cb : g.TNB * 16;
    const int k1 = kr1 - cb < 0 ? 0 : kr1 - cb < kr ? kr1 - cb : kr, k2 = kr - k1;
    const GtStage<VEC, ONE, F32> sv(16 * g.KS, kl, k1, k2);
    const int SR = sv.SR, nth = 64 * g.NG * g.KS, vpt = gt_loads(g.W, VEC);
    if (sv.count() > nth * vpt)
        fail("more vectors than loads", sv.count(), nth, vpt);
    const int nstage = (r1 - r0 + SR - 1) / SR;
    const size_t buf = (size_t)SR * (sv.LDP + sv.RDP) + 32;
    if (2 * buf * sizeof(double) > g.lds)
        fail("stage past the LDS of the launch", SR, sv.LDP, sv.RDP);
    for (int st : {0, 1, 2, 3, nstage / 2, nstage - 2, nstage - 1, nstage, nstage + 1, nstage + 2}) {
        if (st < 0)
            continue;
        const int rows = gt_stage_rows(r1 - r0, SR, st);
        std::vector<char> seen((size_t)SR * (kl + kr), 0);
        for (int t = 0; t < nth; t++)
            for (int u = 0; u < vpt; u++) {
                int c;
                const unsigned info = sv.vector(t + nth * u, c);
                if (gt_row(info) >= rows)
                    continue;
                if (info == ~0u)
                    fail("a lane without a vector loads", st, t, u);
                const int kind = gt_kind(info), row = gt_row(info);
                const int lo = kind == 2 ? k1 : 0, hi = kind == 0 ? kl : kind == 1 ? k1 : kr;
                if (c < lo || c + VEC > hi)
                    fail("column out of range", kind, c, hi);
                if (r0 + (long)st * SR + row >= r1)
                    fail("row out of range", st, row, r1);
                if ((info >> 12) + VEC > buf)
                    fail("LDS offset out of range", (int)(info >> 12), SR, kind);
                for (int e = 0; e < VEC; e++)
                    seen[(size_t)row * (kl + kr) + (kind ? kl : 0) + c + e] = 1;
            }
        const int have = kl + kr - (ONE ? k2 : 0);   // a single column of R2 has its own load
        for (int row = 0; row < rows; row++)
            for (int c = 0; c < have; c++)
                if (!seen[(size_t)row * (kl + kr) + c])
                    fail("not loaded", st, row, c);
    }
}

template <bool F32>
static int all(int n, int kl, int kr1, int kr2)
{
    GramPlan p = plan_gram(n, kl, kr1 + kr2);
    tile_chunks(n, p);
    GramTile g;
    const bool two = plan_pairs(n, kl, kr1, kr2, p, F32, g);
    if (!two)
        g = plan_tile(p.TM, p.TN, 1, p.chunk, p.gx, F32);
    if (!g.NG)
        fail("no plan", n, kl, kr1 + kr2);
    const int gy = (p.TM + g.TMB - 1) / g.TMB * g.nbn;
    for (int x : {0, p.gx / 2, p.gx - 1})
        for (int y = 0; y < gy; y++) {
            const int r0 = x * p.chunk, r1 = n - r0 < p.chunk ? n : r0 + p.chunk;
            if (!two)
                walk<1, false, F32>(g, n, kl, kr1, kr2, r0, r1, y);
            else if (kr2 == 1)
                walk<2, true, F32>(g, n, kl, kr1, kr2, r0, r1, y);
            else
                walk<2, false, F32>(g, n, kl, kr1, kr2, r0, r1, y);
        }
    return two ? 2 : 1;
}

int main(int argc, char **argv)
{
    const int n = atoi(argv[1]), kl = atoi(argv[2]), kr1 = atoi(argv[3]), kr2 = atoi(argv[4]);
    std::printf("ok: %d columns a load, %d with an FP32 R1\n", all<false>(n, kl, kr1, kr2),
                all<true>(n, kl, kr1, kr2));
    return 0;
}
"""


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    d = tmp_path_factory.mktemp("gram_loads")
    (d / "walk.cpp").write_text(WALK)
    kernels = os.path.join(ROOT, "cacg_amd", "csrc", "kernels")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", kernels, str(d / "walk.cpp"), "-o", str(d / "walk")],
                   check=True)
    return str(d / "walk")


# rows: one stage, ragged ends, chunks of fewer and of more rows than a row number of a lane can
# name (1023); columns: few enough to leave lanes without a vector, odd, one, several blocks
@pytest.mark.parametrize("n", [1, 2, 130, 8193, 100003, 600011, 1100000, 2097152, 2147483647])
@pytest.mark.parametrize("kl,kr1,kr2", [(1, 1, 0), (2, 2, 1), (4, 4, 4), (4, 4, 1), (16, 16, 4),
                                        (17, 17, 3), (60, 60, 10), (61, 61, 7), (64, 64, 8),
                                        (99, 99, 11), (127, 127, 0), (128, 129, 17), (256, 256, 32)])
def test_every_load_of_the_tile_kernel_is_in_bounds(walk, n, kl, kr1, kr2):
    r = subprocess.run([walk, str(n), str(kl), str(kr1), str(kr2)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
