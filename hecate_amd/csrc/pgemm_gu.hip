// pgemm_gu.hip - the grouped GEMM's gate/up launches (pgemm.h)
#include "pgemm.h"

using namespace hmoe;

int hmoe::grouped_gate_up(const PgArgs& a, int epi, hipStream_t st)
{
    PgArgs g = a;
    g.ncb = g.shb = 1;
    pg_shared_blocks(g);
    const dim3 grid = pgemm_grid(a.nrb, I / 128, g.nsh);
    if (grid.x == 0) return HMOE_OK;
    g.gx = grid.x;
    if (epi == EPI_ACT) pgemm_kernel<EPI_ACT><<<grid, 256, 0, st>>>(g);
    else pgemm_kernel<EPI_RAW><<<grid, 256, 0, st>>>(g);
    return HMOE_LAUNCHED("grouped gate/up");
}
