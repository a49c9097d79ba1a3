// pgemm_dn.hip - the grouped GEMM's down launches (pgemm.h)
#include "pgemm.h"

using namespace hmoe;

int hmoe::grouped_down(const PgArgs& a, int epi, hipStream_t st)
{
    // Column blocks per workgroup (times are whole moe4p.forward calls, us).
    // Routed: three in one pipeline, since down's k loop is 16 groups and with one column block a third of a workgroup's
    // life is its prologue (256 experts: 150 tokens 843 with one, 823 with three; 1000 tokens 1128, 1108). One where that
    // leaves CUs without a workgroup, which then run three times as long: tables of few experts (8 experts: 450 tokens 71
    // with one, 94 with three; 2048 tokens 116, 154; 48 experts: 187, 192 and 325, 332; from 64 on three again: 244, 237 and
    // 415, 414), or few picks (17 tokens: 96 experts 159, 167; 256 experts 365, 364). Not where the plan has room for many
    // short blocks of them (32 experts, 2048 tokens in blocks of 16, 32 and 64 picks: 3623 with one, 3440 with three; 2212,
    // 2134; 1591, 1564; the room is 32 + picks / block, 160 in blocks of 128: 1193, 1199). Beside the shared expert's blocks the
    // routed ones spread over fewer free slots, and the line is higher (33 tokens: 64 experts 226, 241; 450: 279, 293 and 96
    // experts 400, 409; 128 experts 520, 518).
    // Shared: one, its serial chain over k being the launch's length beside few experts (33 tokens, 8 experts 145 with one,
    // 204 with three; 450 tokens, 32 experts 230, 290; 256 experts, 64 tokens 732, 748). Three in longer chunks beside nearly
    // all experts, where the routed part is several times the chain and the prologues count (256 experts: 150 tokens 875,
    // 875; 300 917, 915; 1000 1223, 1218, uneven 1216, 1208; 2048 1724, 1722; but 176 experts, 2048 tokens 1230, 1238).
    PgArgs g = a;
    g.ncb = a.np < 200 || (a.n_tab < (a.sh0 ? 128 : 64) && a.nrb < 288) ? 1 : 3;
    g.shb = g.ncb == 3 && a.n_tab >= 192 && a.T > 256 ? 3 : 1;
    pg_shared_blocks(g);
    const dim3 grid = pgemm_grid(a.nrb, H / 256 / g.ncb, g.nsh * g.ncb / g.shb);
    if (grid.x == 0) return HMOE_OK;
    g.gx = grid.x;
    if (epi == EPI_D16) pgemm_kernel<EPI_D16><<<grid, 256, 0, st>>>(g);
    else if (epi == EPI_FIN) pgemm_kernel<EPI_FIN><<<grid, 256, 0, st>>>(g);
    else pgemm_kernel<EPI_D><<<grid, 256, 0, st>>>(g);
    return HMOE_LAUNCHED("grouped down");
}
