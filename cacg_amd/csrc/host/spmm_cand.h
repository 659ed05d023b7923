/* The SpMM launch schedules that a solver times on its matrix: of a k-column block,
 * every one another launch.  The default grid (0) is 8192 workgroups up to 32 columns
 * and 4096 above, so each list names the other one; bands, chunks of 1024 to 4096 rows,
 * a resident grid in chunks, and many small workgroups in four sweeps. */
#ifndef CACG_SPMM_CAND_H
#define CACG_SPMM_CAND_H

#include "cacg_kernels.h"

#define SPMM_CANDS 10

static inline cacg_spmm_sched spmm_cand(int k, int i)
{
    static const cacg_spmm_sched narrow[SPMM_CANDS] = {
        {8192, 0, 0},    {4096, 0, 0},   {0, 1024, 0},    {0, 2048, 0},    {0, 4096, 0},
        {4096, 2048, 0}, {768, 2048, 0}, {1024, 1024, 0}, {16384, 512, 4}, {32768, 512, 4}};
    static const cacg_spmm_sched wide[SPMM_CANDS] = {
        {4096, 0, 0},    {8192, 0, 0},   {0, 1024, 0},    {0, 2048, 0},    {0, 4096, 0},
        {8192, 4096, 0}, {768, 2048, 0}, {1024, 1024, 0}, {16384, 512, 4}, {32768, 512, 4}};
    return (k > 32 ? wide : narrow)[i];
}

#endif
