// pgemm_dn.hip - the grouped GEMM's down launches (pgemm.h)
#include "pgemm.h"

using namespace hmoe;

int hmoe::grouped_down(const PgArgs& a, int epi, hipStream_t st)
{
    // A workgroup runs 3 column blocks in one pipeline: down's k loop is 16 groups, so with one column block a third of a
    // workgroup's life is its prologue (150 tokens, 250 experts: 310 us with one, 287 with three). With few picks the
    // launch is a few workgroups per CU and the shorter ones of 2 spread better (17 tokens, 103 experts: 123 against
    // 133 us; equal at about 25 tokens).
    PgArgs g = a;
    g.ncb = a.np < 200 ? 2 : 3;
    pg_shared_blocks(g);
    const dim3 grid(pgemm_grid(a.nrb, H / 256 / g.ncb).x + g.nsh * (H / 256 / g.ncb));
    if (grid.x == 0) return HMOE_OK;
    if (epi == EPI_D16) pgemm_kernel<EPI_D16><<<grid, 256, 0, st>>>(g);
    else if (epi == EPI_FIN) pgemm_kernel<EPI_FIN><<<grid, 256, 0, st>>>(g);
    else pgemm_kernel<EPI_D><<<grid, 256, 0, st>>>(g);
    return HMOE_LAUNCHED("grouped down");
}
