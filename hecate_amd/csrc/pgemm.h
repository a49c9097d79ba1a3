// pgemm.h - the prefill's grouped expert GEMM on gfx950 (runtime/tier/moe4/moe4p.cu:217-245): one launch multiplies
// every row block of the dispatch plan (<= 128 picks of one expert per pass) by that expert's int4 matrices.
//
// Workgroup = (row block, 64 NS output columns of NMAT matrices); 4 waves, each owning 4 weight strips of 16 rows (gate
// and up: 2 of each, down: 4) against all the block's 16-pick tiles, so an input fragment read from LDS feeds 4 MFMAs.
// The tile count NT of a pass is a template parameter picked per block by a uniform switch: the k loop is then
// straight-line code whose registers and LDS follow the block's size, and a small block keeps more bytes in flight
// (what bounds it is the stream of weights from HBM):
//   * weights: 16-byte buffer loads into a ring of D 128-k groups per wave, refilled as each group is consumed (D 4 up to
//     5 tiles; 2 above, where the accumulators need the registers); the row scales 4 groups at a time;
//   * input rows: stages of 64 k by direct global-to-LDS loads into a ring of NBUF stages (8 up to 5 tiles, 4 above;
//     80 KB, so that two workgroups share a CU), issued NBUF - 2 stages before they are read;
//   * each 32-k step's input fragments are read from LDS one step ahead (WN tiles ahead above 5 tiles), each read issued
//     behind the MFMAs that free its registers.
// Every load is one the compiler sees (the stage ring is eight separate LDS arrays at compile-time indices, so that it
// can tell a stage being filled from the one being read), so its waits count exactly and no wait drains the rings. The
// one wait placed by hand is a wave's own stage loads before the barrier that publishes them; the loads after a stage in
// program order are fixed (sched_barrier around each bundle), so that count is a compile-time constant too.
//
// Measured on one layer of 256 experts, the shared expert included, whole moe4p.forward calls against the same tiles with
// two 128-k stages, a 2-deep weight ring whose waits also waited for the stage loads, and the shared expert in launches of
// its own (bits equal): 33 tokens 688 -> 565 us, 150 tokens 1046 -> 871, 450 1145 -> 975, 1000 1366 -> 1232, 2048 1786 ->
// 1736. At 33 to ~500 tokens the weight stream bounds it (33 tokens, without the shared expert: 3.1 GB of 165 experts in 528
// us, 5.9 TB/s; a read-only stream reaches 6.05). At 2048 the issue slots (counters of the gate/up launch, per SIMD): 976 K
// cycles of MFMA and 700 K of other VALU, mostly the 13 instructions a fragment costs to dequantise, in a launch of 1930 K,
// at a clock the power limit holds at 1.6-1.9 GHz; waits on loads are 0.14 of the wave cycles, waits to issue 0.52. At 1000
// tokens of uneven popularity neither is full: 531 K and 592 K of 1496 K cycles, and 4.3 TB/s. An epilogue chosen at run
// time instead of by template spills registers in the k loop (+5 to 8 %).
#pragma once
#include "hmoe_dev.h"

namespace hmoe {

constexpr int PG_PB = 128;                  // picks per pass
constexpr int PG_STL = 5;                   // 16-pick tiles per stage array
constexpr int PG_SA = PG_STL * 128;         // u32x4 per stage array (2 KB per tile)

enum { EPI_ACT = 0, EPI_RAW = 1, EPI_D = 2, EPI_FIN = 3, EPI_D16 = 4 };

struct Block { int e, p0, rows; };

// The workgroup's row block and column block. The dispatcher deals a launch's workgroups round-robin over the 8
// XCDs (workgroup i runs on XCD i % 8), each with its own L2: the column blocks of one row block go to consecutive
// workgroups of one XCD, so they run together and read the block's input rows from that XCD's L2 (one fetch from
// memory instead of one per column block). i: the workgroup's index among nrb (rounded up to 8) x ny.
__device__ __forceinline__ void xcd_tile(int i, int& rb, int& cb, int ny)
{
    const int j = i >> 3;
    rb = (j / ny) * 8 + (i & 7);
    cb = j % ny;
}

// The grid of nrb row blocks x ny column blocks and extra x ny workgroups more, and a workgroup's index in it. Two
// dimensions: a launch's x extent is at most 2^32 threads, which a plan of 524,288 blocks would pass in one. (x the extent
// from the launch's own arguments: gridDim reads the dispatch packet, a round trip to the queue's memory at every workgroup
// start)
inline dim3 pgemm_grid(int nrb, int ny, int extra = 0) { return dim3(((nrb + 7) & ~7) + extra, ny); }
__device__ __forceinline__ int pgemm_index(int gx) { return blockIdx.x + gx * blockIdx.y; }

// a scalar load from memory that no kernel of the launch writes: under the weight stream a vector load returns behind
// every load the CU has in flight (over 1 us), a scalar load does not wait for them. The address must be the same in
// every lane.
template <typename T> __device__ __forceinline__ T ld_uniform(const T* p)
{
    return *(const __attribute__((address_space(4))) T*) p;
}

// row block rb of the plan: up to 256 picks (the dispatch's bm <= 256), run as passes; a block whose expert or picks fall
// outside the tables (np picks) is skipped, so a caller's malformed plan reads nothing out of bounds
__device__ __forceinline__ bool get_block(const int* rbt, int nrb, const int* meta, int n_tab, int np, int rb, Block& b)
{
    if (rb >= nrb || (meta && rb >= ld_uniform(meta + 1))) return false;
    b.e = ld_uniform(rbt + 4 * rb);
    b.p0 = ld_uniform(rbt + 4 * rb + 1);
    b.rows = min(ld_uniform(rbt + 4 * rb + 2), 256);
    return b.e >= 0 && b.e < n_tab && b.rows > 0 && b.p0 >= 0 && b.p0 <= np - b.rows;
}

// one launch of the grouped GEMM. Gate/up (NMAT 2): xin = f16 x [T][H], row of pick p tok[p] (tok NULL: p itself); down
// (NMAT 1): xin = act rows [np][I]. Epilogues (epi): gate/up -> act f16 ar = silu(g) u wt (EPI_ACT) or the raw gate and
// up sums (EPI_RAW, fp32 [2][ps][I], the test entry of moe4t); down -> f16 rows for the ordered combine (EPI_D16), fp32
// rows (EPI_D, the moe4t.gemm test entry) or added into out[tok] with fp32 atomics (EPI_FIN, moe4t.cu's down epilogue)
struct PgArgs
{
    const _Float16* xin;
    const int* tok;
    const float* wt;
    const int* rbt;
    const int* meta;
    const int64_t* w0;
    const int64_t* w1;
    const int64_t* s0;
    const int64_t* s1;
    void* out;
    int nrb, n_tab, T, np, ps;
    int ncb, shb;                           // column blocks per workgroup: routed, shared (set by the launchers)
    // the shared expert (row-major f16 [N][K], NULL: none) on every one of the T tokens in the same launch: its rows follow
    // the picks' (row ps + t of the act, and of down's rows)
    const _Float16* sh0;
    const _Float16* sh1;
    int nsh, sh_rows;                       // its token blocks and the tokens of each (set by the launchers)
    int gx;                                 // the grid's x extent (set by the launchers)
};
// the shared expert's token blocks: of equal size, whole tiles, at most PG_PB
inline void pg_shared_blocks(PgArgs& a)
{
    a.nsh = a.sh0 ? (a.T + PG_PB - 1) / PG_PB : 0;
    a.sh_rows = a.nsh ? (((a.T + a.nsh - 1) / a.nsh) + 15) & ~15 : 0;
}
int grouped_gate_up(const PgArgs& a, int epi, hipStream_t st);
int grouped_down(const PgArgs& a, int epi, hipStream_t st);

__device__ __forceinline__ __amdgpu_buffer_rsrc_t pg_rsrc(uint64_t p, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc((void*) p, (short) 0, (int) bytes, 0x00020000);
}

// 16 bytes per lane from a buffer to LDS (lane l at lds + 16 l). (Device pass only: the host target knows no 16-byte form.)
__device__ __forceinline__ void pg_load_lds(__amdgpu_buffer_rsrc_t rs, u32x4* lds, uint32_t voff, int soff)
{
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*) lds, 16, (int) voff, soff, 0, 0);
#endif
}

// the epilogue of a pass: lane holds output rows n .. n + 4 of pick pk (row p0 + pk of the output). SH: the shared expert's
// (weight 1)
template <int EPI, int NT, bool SH>
__device__ __forceinline__ void pg_store(const PgArgs& a, int p0, int rows, int nb0, int lane, const f32x4 (&acc)[4][NT])
{
    constexpr int NMAT = EPI == EPI_ACT || EPI == EPI_RAW ? 2 : 1, NS = 4 / NMAT, NOUT = NMAT == 2 ? I : H;
    // (an opaque copy of the lane: no address formed here is kept in registers across the k loop)
    int l;
    asm volatile("v_mov_b32 %0, %1" : "=v"(l) : "v"(lane));
    #pragma unroll
    for (int tt = 0; tt < NT; ++tt)
    {
        const int pk = tt * 16 + (l & 15);
        if (pk >= rows) continue;
        const size_t p = (size_t) p0 + pk;
        const float wv = EPI == EPI_ACT && !SH ? a.wt[p] : 1.f;
        const int tk = EPI == EPI_FIN ? a.tok[p] : 0;
        #pragma unroll
        for (int st = 0; st < NS; ++st)
        {
            const int n = (nb0 + st) * 16 + 4 * (l >> 4);
            if (NMAT == 2)
            {
                const f32x4 g = acc[2 * st][tt], u = acc[2 * st + NMAT - 1][tt];
                if (EPI == EPI_ACT)
                {
                    _Float16 o[4];
                    #pragma unroll
                    for (int i = 0; i < 4; ++i) o[i] = (_Float16) (silu(g[i]) * u[i] * wv);
                    *(uint2*) ((_Float16*) a.out + p * NOUT + n) = *(const uint2*) o;
                }
                else
                {
                    *(f32x4*) ((float*) a.out + p * NOUT + n) = g;
                    *(f32x4*) ((float*) a.out + ((size_t) a.ps + p) * NOUT + n) = u;
                }
            }
            else
            {
                const f32x4 d = acc[st][tt];
                if (EPI == EPI_D16)
                {
                    // (a pick's down row rounded to f16: half the bytes written here and read by the combine)
                    _Float16 o[4];
                    #pragma unroll
                    for (int i = 0; i < 4; ++i) o[i] = (_Float16) d[i];
                    *(uint2*) ((_Float16*) a.out + p * NOUT + n) = *(const uint2*) o;
                }
                else if (EPI == EPI_FIN)
                {
                    // out[tok] += d (the combine in the epilogue, fp32 atomics as moe4t.cu's down GEMM: no d buffer)
                    if ((unsigned) tk < (unsigned) a.T)
                    {
                        float* o = (float*) a.out + (size_t) tk * NOUT + n;
                        #pragma unroll
                        for (int i = 0; i < 4; ++i) unsafeAtomicAdd(o + i, d[i]);
                    }
                }
                else *(f32x4*) ((float*) a.out + p * NOUT + n) = d;
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// The input rows of a pass, staged in LDS as f16. A stage holds each tile's 16 rows x 64 k as two 1 KB blocks (row
// halves): lane l of a block's load takes row l / 8's 16-byte chunk (l % 8) ^ (l / 8) (whole 128-byte lines from memory)
// and lands at 16 l, so a fragment read (row l % 16, chunk 4 k + l / 16) meets distinct banks. Wave w loads half w % 2 of
// tiles 2 j + w / 2; a pick past the block re-reads its last row (its output columns are never stored), a tile past it the
// last tile.
template <int NMAT, int NT, int NBUF, typename BUF>
struct PgIn
{
    static constexpr int K = NMAT == 2 ? H : I, KS = K / 64, ND = (NT + 1) / 2;       // ND: stage loads per wave
    BUF buf;
    __amdgpu_buffer_rsrc_t xrs;
    uint32_t src[ND];
    int fo[2], w;

    // row(p): the input row of pick p of the pass
    template <typename ROW>
    __device__ __forceinline__ void init(__amdgpu_buffer_rsrc_t x, int rows, ROW&& row_of)
    {
        const int l = threadIdx.x & 63, row = l & 15, ntt = (rows + 15) >> 4;
        w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        xrs = x;
        #pragma unroll
        for (int j = 0; j < ND; ++j)
        {
            const int pk = min(min(2 * j + (w >> 1), ntt - 1) * 16 + 8 * (w & 1) + (l >> 3), rows - 1);
            src[j] = (uint32_t) row_of(pk) * (K * 2) + 16 * ((l & 7) ^ (l >> 3));
        }
        #pragma unroll
        for (int k = 0; k < 2; ++k) fo[k] = (row >> 3) * 64 + 8 * (l & 7) + ((4 * k + (l >> 4)) ^ (l & 7));
    }
    // input stage s (of a column block's KS; past the last it wraps into the next column block's) into ring buffer J: one
    // array per buffer, or (4 buffers) two, tiles 4 .. in the second
    template <int J> __device__ __forceinline__ void stage(int s)
    {
        const int so = (s >= KS ? s - KS : s) * 128;
        #pragma unroll
        for (int j = 0; j < ND; ++j)
        {
            const int tt = min(2 * j + (w >> 1), NT - 1);
            auto put = [&](u32x4* arr, int tl) {
                pg_load_lds(xrs, arr + (tl * 2 + (w & 1)) * 64, src[j], so);
            };
            if constexpr (NBUF == 8) put(buf(ic<J>{}), tt);
            else { if (2 * j < 4) put(buf(ic<2 * J>{}), tt); else put(buf(ic<2 * J + 1>{}), tt - 4); }
        }
    }
    // fragment of tile i, 32-k step k of ring buffer J
    template <typename JC> __device__ __forceinline__ f16x8 rd(JC, int i, int k)
    {
        constexpr int J = JC::value;
        if constexpr (NBUF == 8) return as_f16x8(buf(ic<J>{})[i * 128 + fo[k]]);
        else return i < 4 ? as_f16x8(buf(ic<2 * J>{})[i * 128 + fo[k]]) : as_f16x8(buf(ic<2 * J + 1>{})[(i - 4) * 128 + fo[k]]);
    }
};

// one pass: the picks of b (<= 16 NT) against column blocks cb0 .. cb0 + ncb of 64 NS columns, one continuous pipeline
// (the next column block's weights and input stages load under the last groups of the one before)
template <int EPI, int NT, int D, typename BUF>
__device__ __forceinline__ void pg_pass(BUF buf, const PgArgs& a, const Block& b, int cb0, int ncb_)
{
    constexpr int NMAT = EPI == EPI_ACT || EPI == EPI_RAW ? 2 : 1;
    const int ncb = NMAT == 2 ? 1 : ncb_;                   // (gate/up: one, which frees the rings for its epilogue)
    constexpr int K = NMAT == 2 ? H : I, NOUT = NMAT == 2 ? I : H, KG = K / 128, KS = K / 64, NS = 4 / NMAT;
    constexpr int NBUF = NT <= PG_STL ? 8 : 4;              // input stages in LDS
    constexpr int WN = NT == 8 ? 2 : NT == 7 ? 4 : NT == 6 ? 3 : NT;      // input fragments held
    constexpr int ND = (NT + 1) / 2;
    static_assert(WN <= NT && 16 * NT % WN == 0 && KS % 8 == 0 && (D == 2 || D == 4), "the loop is unrolled over 8 stages");
    const int t = threadIdx.x, l = t & 63, row = l & 15;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);   // wave index, kept in a scalar register
    const int nb0 = (cb0 * 4 + w) * NS;
    const DqConsts dq = dq_consts();
    PgIn<NMAT, NT, NBUF, BUF> in = {buf};
    in.init(pg_rsrc((uint64_t) a.xin, (uint32_t) (NMAT == 2 ? a.T : a.np) * (K * 2)), b.rows, [&](int pk) {
        int r = b.p0 + pk;
        if (NMAT == 2)
        {
            if (a.tok) r = a.tok[r];
            r = (unsigned) r < (unsigned) a.T ? r : 0;
        }
        return r;
    });
    auto stage = [&](int s, auto jc) { in.template stage<decltype(jc)::value>(s); };
    auto rd = [&](auto jc, int i, int k) { return in.rd(jc, i, k); };
    __amdgpu_buffer_rsrc_t wrs[NMAT], srs[NMAT];
    #pragma unroll
    for (int m = 0; m < NMAT; ++m)
    {
        wrs[m] = pg_rsrc((uint64_t) ld_uniform((m == 0 ? a.w0 : a.w1) + b.e), NOUT * (K / 2));
        srs[m] = pg_rsrc((uint64_t) ld_uniform((m == 0 ? a.s0 : a.s1) + b.e), NOUT * KG * 2);
    }
    // the weights of group g (counted through the column blocks; past the last one its last group again) into ring slot
    // SL; when g starts a block of 4, the block's row scales too (a block's 4 bf16 of one row are 8 contiguous bytes of
    // I4G128) into sc4[SC] (SC -1: none)
    u32x4 ring[D][4];
    u32x2 sc4[2][4];
    auto fetch = [&](int g, auto sl, auto sc) {
        constexpr int SL = decltype(sl)::value, SC = decltype(sc)::value;
        const int gc = min(g, ncb * KG - 1), c = gc / KG, gk = gc - c * KG;
        #pragma unroll
        for (int f = 0; f < 4; ++f)
        {
            const int nb = nb0 + c * (4 * NS) + f / NMAT;
            ring[SL][f] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrs[f % NMAT], l * 16,
                                                                                     (nb * KG + gk) * 1024, 2));
            if constexpr (SC >= 0)
                sc4[SC][f] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(srs[f % NMAT], row * 8,
                                                                     (nb * (KG / 4) + (gk >> 2)) * 128, 0));
        }
    };
    f32x4 acc[4][NT];
    auto clear = [&]() {
        #pragma unroll
        for (int f = 0; f < 4; ++f)
            #pragma unroll
            for (int i = 0; i < NT; ++i) acc[f][i] = (f32x4) {0.f, 0.f, 0.f, 0.f};
    };
    static_for<D>([&](auto g) {
        constexpr int G = decltype(g)::value;
        fetch(G, g, ic<G == 0 ? 0 : -1>{});
        __builtin_amdgcn_sched_barrier(0);
    });
    static_for<NBUF - 1>([&](auto j) {
        stage(decltype(j)::value, j);
        __builtin_amdgcn_sched_barrier(0);
    });
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    f16x8 bq[WN];
    #pragma unroll
    for (int i = 0; i < WN; ++i) bq[i] = rd(ic<0>{}, i, 0);
    for (int c = 0; c < ncb; ++c)
    {
        clear();
        for (int s0 = 0; s0 < KS; s0 += 8)
        {
        static_for<8>([&](auto sc8) {
            constexpr int s8 = decltype(sc8)::value, G = s8 / 2, SL = G % D;
            constexpr int J0 = s8 % NBUF, J1 = (s8 + 1) % NBUF, JL = (s8 + NBUF - 1) % NBUF;    // ring buffers
            static_for<2>([&](auto kc) {
                constexpr int k = decltype(kc)::value, kq = 2 * (s8 & 1) + k;       // 32-k step of the group
                f16x8 aw[4];
                #pragma unroll
                for (int f = 0; f < 4; ++f)
                {
                    const uint32_t sw = sc4[0][f][G / 2];                           // bf16 of the group: half G % 2
                    const _Float16 h = (_Float16) __uint_as_float(G % 2 == 0 ? sw << 16 : sw & 0xffff0000u);
                    aw[f] = dq8s(ring[SL][f][kq], (f16x2) {h, h}, dq);
                }
                if constexpr (k == 1)
                {
                    // publish the next stage: this wave's loads of it are older than the bundles after the one that
                    // issued it, NBUF - 1 stages ago (ND stage loads each, and on odd stages a ring refill: 4 weight
                    // loads and, when it starts a block of 4 groups, 4 scale loads). The stage whose buffer the next
                    // loads take was last read before the previous barrier.
                    __builtin_amdgcn_sched_barrier(0);
                    constexpr int after = [] {
                        int n = 0;
                        for (int q = s8 + 3 - NBUF; q <= s8 - 1; ++q)
                        {
                            const int qq = (q + 16) % 8;
                            n += ND;
                            if (qq & 1) n += (qq / 2 + D) % 4 == 0 ? 8 : 4;
                        }
                        return n;
                    }();
                    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(after) : "memory");
                    __builtin_amdgcn_s_barrier();
                    __builtin_amdgcn_sched_barrier(0);
                    stage(s0 + s8 + NBUF - 1, ic<JL>{});
                    // on odd stages the group's ring slot is consumed: refill it D groups ahead
                    if constexpr (s8 & 1) fetch(c * KG + s0 / 2 + G + D, ic<SL>{}, ic<(G + D) % 4 == 0 ? 1 : -1>{});
                    __builtin_amdgcn_sched_barrier(0);
                }
                #pragma unroll
                for (int i = 0; i < NT; ++i)
                {
                    // (fragments take the window's slots in turn, across the 16 steps of the unrolled loop)
                    const int q = ((2 * s8 + k) * NT + i) % WN;
                    #pragma unroll
                    for (int f = 0; f < 4; ++f) acc[f][i] = mfma16(aw[f], bq[q], acc[f][i]);
                    // the fragment WN tiles on: of this step, or of the next one
                    if (i + WN < NT) bq[q] = rd(ic<J0>{}, i + WN, k);
                    else bq[q] = k == 0 ? rd(ic<J0>{}, i + WN - NT, 1) : rd(ic<J1>{}, i + WN - NT, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            });
            if constexpr (s8 == 7)
            {
                #pragma unroll
                for (int f = 0; f < 4; ++f) sc4[0][f] = sc4[1][f];
            }
        });
        }
        pg_store<EPI, NT, false>(a, b.p0, b.rows, nb0 + c * (4 * NS), l, acc);
    }
    // (no stage load may land in LDS after the workgroup has given it up)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// A pass of the shared expert, merged into the routed launches: by itself it was two dense launches whose few workgroups
// were a chain of 96 and 32 serial stages (83 + 25 us from 17 to ~500 tokens, 104 + 64 at 2048); here that chain runs beside
// the routed blocks (33 tokens: 706 -> 639 us per layer; 150: 993 -> 935; 1000: 1311 -> 1263; 2048: 1815 -> 1796).
// tokens t0 .. t0 + rows (<= 16 NT) against column blocks cb0 .. cb0 + ncb. As pg_pass with the
// f16 weights loaded as fragments (16 rows x 64 bytes) into a ring of DS 64-k stages, each refilled one step after its
// last use; the k order of every sum is that of a 32-k chain, as everywhere.
template <int EPI, int NT, int DS, typename BUF>
__device__ __forceinline__ void pg_dense(BUF buf, const PgArgs& a, int t0, int rows, int cb0, int ncb_)
{
    constexpr int NMAT = EPI == EPI_ACT ? 2 : 1;
    const int ncb = NMAT == 2 ? 1 : ncb_;
    constexpr int K = NMAT == 2 ? H : I, NOUT = NMAT == 2 ? I : H, KS = K / 64, NS = 4 / NMAT;
    constexpr int NBUF = NT <= PG_STL ? 8 : 4, WN = NT > 6 ? 2 : NT > 5 ? 3 : NT, ND = (NT + 1) / 2;
    static_assert(NT % WN == 0 && KS % 8 == 0 && 8 % DS == 0, "the loop is unrolled over 8 stages");
    const int l = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nb0 = (cb0 * 4 + w) * NS, r0 = NMAT == 2 ? t0 : a.ps + t0;                // first input row
    PgIn<NMAT, NT, NBUF, BUF> in = {buf};
    in.init(pg_rsrc((uint64_t) a.xin, (uint32_t) (NMAT == 2 ? a.T : a.ps + a.T) * (K * 2)), rows,
            [&](int pk) { return r0 + pk; });
    auto stage = [&](int s, auto jc) { in.template stage<decltype(jc)::value>(s); };
    auto rd = [&](auto jc, int i, int k) { return in.rd(jc, i, k); };
    __amdgpu_buffer_rsrc_t wrs[NMAT];
    #pragma unroll
    for (int m = 0; m < NMAT; ++m) wrs[m] = pg_rsrc((uint64_t) (m == 0 ? a.sh0 : a.sh1), NOUT * K * 2);
    const int wo = (l & 15) * (K * 2) + 16 * (l >> 4);
    // the weights of stage s (counted through the column blocks; past the last one its last stage again) into slot SL
    u32x4 ring[DS][2][4];
    auto fetch = [&](int s, auto sl) {
        constexpr int SL = decltype(sl)::value;
        const int sc = min(s, ncb * KS - 1), c = sc / KS, sk = sc - c * KS;
        #pragma unroll
        for (int k = 0; k < 2; ++k)
            #pragma unroll
            for (int f = 0; f < 4; ++f)
                ring[SL][k][f] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrs[f % NMAT], wo,
                    (nb0 + c * (4 * NS) + f / NMAT) * (16 * K * 2) + (2 * sk + k) * 64, 0));
    };
    f32x4 acc[4][NT];
    static_for<DS - 1>([&](auto g) {
        fetch(decltype(g)::value, g);
        __builtin_amdgcn_sched_barrier(0);
    });
    static_for<NBUF - 1>([&](auto j) {
        stage(decltype(j)::value, j);
        __builtin_amdgcn_sched_barrier(0);
    });
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    f16x8 bq[WN];
    #pragma unroll
    for (int i = 0; i < WN; ++i) bq[i] = rd(ic<0>{}, i, 0);
    for (int c = 0; c < ncb; ++c)
    {
        #pragma unroll
        for (int f = 0; f < 4; ++f)
            #pragma unroll
            for (int i = 0; i < NT; ++i) acc[f][i] = (f32x4) {0.f, 0.f, 0.f, 0.f};
        for (int s0 = 0; s0 < KS; s0 += 8)
            static_for<8>([&](auto sc8) {
                constexpr int s8 = decltype(sc8)::value, SL = s8 % DS;
                constexpr int J0 = s8 % NBUF, J1 = (s8 + 1) % NBUF, JL = (s8 + NBUF - 1) % NBUF;
                static_for<2>([&](auto kc) {
                    constexpr int k = decltype(kc)::value;
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (k == 0) fetch(c * KS + s0 + s8 + DS - 1, ic<(s8 + DS - 1) % DS>{});
                    else
                    {
                        // the next stage, as in pg_pass: older than the stage loads of the last NBUF - 3 bundles and the 8
                        // weight loads of each of the last NBUF - 2 stages
                        asm volatile("s_waitcnt vmcnt(%0)" :: "n"((NBUF - 3) * ND + (NBUF - 2) * 8) : "memory");
                        __builtin_amdgcn_s_barrier();
                        __builtin_amdgcn_sched_barrier(0);
                        stage(s0 + s8 + NBUF - 1, ic<JL>{});
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    #pragma unroll
                    for (int i = 0; i < NT; ++i)
                    {
                        #pragma unroll
                        for (int f = 0; f < 4; ++f) acc[f][i] = mfma16(as_f16x8(ring[SL][k][f]), bq[i % WN], acc[f][i]);
                        if (i + WN < NT) bq[i % WN] = rd(ic<J0>{}, i + WN, k);
                        else bq[i % WN] = k == 0 ? rd(ic<J0>{}, i + WN - NT, 1) : rd(ic<J1>{}, i + WN - NT, 0);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                });
            });
        pg_store<EPI, NT, true>(a, a.ps + t0, rows, nb0 + c * (4 * NS), l, acc);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

template <int EPI>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) pgemm_kernel(PgArgs a)
{
    __shared__ __attribute__((aligned(16))) u32x4 b0[PG_SA], b1[PG_SA], b2[PG_SA], b3[PG_SA], b4[PG_SA], b5[PG_SA],
        b6[PG_SA], b7[PG_SA];
    auto buf = [&](auto jc) -> u32x4* {
        constexpr int J = decltype(jc)::value;
        if constexpr (J == 0) return b0;
        else if constexpr (J == 1) return b1;
        else if constexpr (J == 2) return b2;
        else if constexpr (J == 3) return b3;
        else if constexpr (J == 4) return b4;
        else if constexpr (J == 5) return b5;
        else if constexpr (J == 6) return b6;
        else return b7;
    };
    constexpr int NMAT = EPI == EPI_ACT || EPI == EPI_RAW ? 2 : 1;
    constexpr int NCB = (NMAT == 2 ? I : H) / (256 / NMAT);
    const int ny = NCB / a.ncb;
    int i = pgemm_index(a.gx);
    if constexpr (EPI == EPI_ACT || EPI == EPI_D16)
    {
        // the shared expert's blocks come first: they are the longest, and the rest fills in around them. The token blocks of
        // one column block go to consecutive workgroups of one XCD, which then reads its weights once (NCB / shb is a
        // multiple of 8: 16 in gate/up, 24 or 8 in down, where shb divides ncb).
        const int ns = a.nsh * (NCB / a.shb);
        if (i < ns)
        {
            const int j = i >> 3;
            const int cb = (j / a.nsh) * 8 + (i & 7), t0 = j % a.nsh * a.sh_rows, rows = min(a.sh_rows, a.T - t0);
            if (rows <= 0) return;
            switch ((rows + 31) >> 5)
            {
                case 1: pg_dense<EPI, 2, 4>(buf, a, t0, rows, cb * a.shb, a.shb); break;
                case 2: pg_dense<EPI, 4, 4>(buf, a, t0, rows, cb * a.shb, a.shb); break;
                case 3: pg_dense<EPI, 6, 2>(buf, a, t0, rows, cb * a.shb, a.shb); break;
                default: pg_dense<EPI, 8, 2>(buf, a, t0, rows, cb * a.shb, a.shb); break;
            }
            return;
        }
        i -= ns;
    }
    int rbi, cbi;
    xcd_tile(i, rbi, cbi, ny);
    Block rb;
    if (!get_block(a.rbt, a.nrb, a.meta, a.n_tab, a.np, rbi, rb)) return;
    // a block of more than PG_PB picks runs as passes, one after the other (a later pass reads the weights again,
    // mostly from the caches); the barrier between them keeps one pass's last LDS reads ahead of the next pass's loads
    for (int h0 = 0; h0 < rb.rows; h0 += PG_PB)
    {
        if (h0) __syncthreads();
        const Block b = {rb.e, rb.p0 + h0, min(PG_PB, rb.rows - h0)};
        switch ((b.rows + 15) >> 4)
        {
            case 1: pg_pass<EPI, 1, 4>(buf, a, b, cbi * a.ncb, a.ncb); break;
            case 2: pg_pass<EPI, 2, 4>(buf, a, b, cbi * a.ncb, a.ncb); break;
            case 3: pg_pass<EPI, 3, 4>(buf, a, b, cbi * a.ncb, a.ncb); break;
            case 4: pg_pass<EPI, 4, 4>(buf, a, b, cbi * a.ncb, a.ncb); break;
            case 5: pg_pass<EPI, 5, 4>(buf, a, b, cbi * a.ncb, a.ncb); break;
            case 6: pg_pass<EPI, 6, 2>(buf, a, b, cbi * a.ncb, a.ncb); break;
            case 7: pg_pass<EPI, 7, 2>(buf, a, b, cbi * a.ncb, a.ncb); break;
            default: pg_pass<EPI, 8, 2>(buf, a, b, cbi * a.ncb, a.ncb); break;
        }
    }
}

}  // namespace hmoe
