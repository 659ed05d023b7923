"""The launch schedules the solvers time (host side, no GPU): each another launch, and none of those
left out that some matrix may want."""

import os
import subprocess

import pytest

from conftest import ROOT

PRINT = r"""
#include <stdio.h>
#include <stdlib.h>
#include "spmm_cand.h"
int main(int argc, char **argv)
{
    const int k = atoi(argv[1]), base = k > 32 ? 4096 : 8192;
    for (int i = 0; i < SPMM_CANDS; i++) {
        const cacg_spmm_sched s = spmm_cand(k, i);
        printf("%d %d %d\n", s.grid ? s.grid : base, s.chunk_rows, s.passes);
    }
    return 0;
}
"""


@pytest.fixture(scope="module")
def show(tmp_path_factory):
    d = tmp_path_factory.mktemp("spmm_cand")
    (d / "show.c").write_text(PRINT)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["gcc", "-std=gnu11", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(rocm, "include"),
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "cacg_amd/csrc/host"),
                    str(d / "show.c"), "-o", str(d / "show")], check=True)
    return str(d / "show")


@pytest.mark.parametrize("k", [1, 4, 16, 32, 33, 64, 128])
def test_candidates_are_distinct_launches_and_complete(show, k):
    out = subprocess.run([show, str(k)], check=True, capture_output=True, text=True).stdout
    got = [tuple(map(int, l.split())) for l in out.splitlines()]
    assert len(got) == len(set(got))
    grid = 4096 if k > 32 else 8192
    bands = [(4096, 0, 0), (8192, 0, 0)]
    chunks = [(grid, c, 0) for c in (1024, 2048, 4096)]
    assert set(bands + chunks + [(16384, 512, 4), (32768, 512, 4), (768, 2048, 0), (1024, 1024, 0)]) <= set(got)
