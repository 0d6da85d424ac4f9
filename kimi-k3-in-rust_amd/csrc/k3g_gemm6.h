/* k3g_gemm6.h - the routed experts' products for many tokens as grouped GEMMs on the scaled
 * FP4 x FP6 matrix instructions (v_mfma_scale_f32_16x16x128_f8f6f4, fp32 accumulation).
 *
 * The engine computes, per (token, slot) pair, three MXFP4 GEMVs per expert in its
 * moe_prefill_chunk loop (src/core/k3_ops.c:668-808); here the pairs are grouped by expert (the
 * stable counting sort of k3g_misc.hip) and each expert's pairs are the columns of one GEMM:
 *
 *   gate/up  (mode 0):  G = W1 X, U = W3 X  -> h = act(G, U)   (K = hidden, or latent)
 *   down     (mode 1):  Y = W2 h            -> contrib rows    (K = inter)
 *
 * Operands. The weights are the A operand exactly as the tiled MXFP4 layout stores them: FP4
 * codes and their E8M0 scales, never decoded. An activation is the sum of four FP6 (E2M3)
 * pieces, each with its own E8M0 scale per 32 values (v = p0 + r, r = p1 + r', ...): what is
 * left after four is 6.6e-7 of normally distributed values (2-norm; 9e-7 for silu(g) u), where two
 * bf16 pieces leave 2.5e-6 and a bf16 piece with an MXFP8 remainder 3.9e-5. But it is 3e-7 of the
 * block's largest value, at most 2^-16 of it, for each of its values: a block whose values lie far
 * below its largest takes eight pieces (gm_eight). FP4 x FP6 runs at
 * the FP4 rate (8.7 PFLOP/s measured, bf16 2.35), so four pieces cost what one bf16 piece
 * does, and 128 products of E2M1 and E2M3 sum exactly before they are added to the fp32
 * accumulator (FP4 x FP8 does not: 2e-5).
 *
 * Activation rows ("quads"): per row and 512 columns 1664 bytes, 13 lines of 128: for each of
 * the four 128-column steps j 384 bytes, dwords 0 .. 3 of piece p of the step's 32-column block q
 * at 64 p + 16 q, then dwords 4 and 5 at 256 + 32 p + 8 q; and a line of scales, dword 4 j + q
 * the four pieces' bytes of step j's block q. The second four pieces of a block lie in a second
 * array of quads, all rows after the first; a scale dword of zero there: the block has none.
 *
 * Work unit: one workgroup of 4 waves = (up to 64 pairs of a column tile, 512 or 256 weight
 * rows: half gate and the same up rows, or output rows). Wave w owns 16 RG rows (RG = 8 or 4)
 * and all NB column blocks of 16. Its weights go from HBM to registers, two steps ahead;
 * the activations are copied to LDS ahead by global_load_lds_dwordx4, eight columns
 * x one whole line per instruction (instructions that took 64 bytes of 16 columns met the
 * other half of each line still on its way: the cache stalls on that, and 49-75 % of its
 * cycles went there), the 16-byte units of column c swizzled by c % 8 so that the B-operand
 * reads meet no bank conflict. Two workgroups run per CU, so one's matrix work covers the
 * other's barrier and waits. The items with a row that has blocks of eight pieces go through those
 * blocks' steps once more, with the second array: gate/up of 4,096 tokens 1.66 -> 4.4 ms with such
 * blocks everywhere, 2.28 -> 3.0 everywhere in one token of 50.
 *
 * What bounds it: with 1 and 2 column blocks the weight stream (gate/up of 256 tokens of the K2
 * layer, 6.0 GB, 0.93 ms, 6.4 TB/s); with full tiles the matrix cores, which hold 1.7 GHz on FP6
 * data (gate/up of 32,768 pairs in full tiles 1.73 ms, 1.11 PFLOP/s; on two bf16 pieces it
 * took 2.58; down 0.99, as bf16 + MXFP8 remainder 1.27-1.30). K3, 2,000 tokens (896 experts of
 * about 36 pairs): gate/up 4.33 -> 3.01 ms beside the shared expert; K2, 4,096 bf16 tokens: down
 * 1.68 -> 1.40.
 *
 * Workgroup order: k3g_gemm.hip's (tiles largest first, dealt to the XCDs in groups). */
#pragma once

#include "k3g_gemm.h"

#define G6_ROWS 256                 /* weight rows per workgroup (twice that with RG = 8) */
#define G6_QB K3G_P6_QUAD           /* bytes of one activation quad */
#define G6_BLK (6 * 1024)           /* a step of one column block in LDS */
#define G6_LDS (72 * 1024)          /* 2 stages of 4 blocks or 3 of 3, 2 quads of their scales; the epilogue
                                     * takes all of it */
#define G6_LIST (63 * 1024)         /* the steps of g6_again (9 KB: K to 589,824) */
#define G6_BIG_MIN 1024             /* workgroups from which on RG = 8 (g6_setup) */
#define G6_QT 4352                  /* tiled MXFP4 quad tile */

/* x (fp32 [T][K]) -> activation quads, a workgroup per row, one thread per block of 32; the blocks
 * of the last 128-column step past K are zero. wrow[t]: row t has blocks of eight pieces; *wide is
 * then raised. V4: x is 16-byte aligned. Nothing when *run_flag is 0. */
template <bool V4>
__global__ void __launch_bounds__(256)
k_x6(const float *__restrict__ x, int K, uint8_t *__restrict__ o, size_t more,
     uint8_t *__restrict__ wrow, int32_t *__restrict__ wide, const int32_t *__restrict__ run_flag)
{
    if (run_flag && !*run_flag) return;
    const int nbk = 4 * ((K + 127) / 128), nQ = (K + 511) / 512, t = blockIdx.x;
    bool any = false;
    for (int k = threadIdx.x; k < nbk; k += blockDim.x) {
        gm_v16f ev = {}, od = {};
        if (32 * k < K) {
            const float *p = x + (size_t)t * K + 32 * k;
            if (V4) {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float4 v = ((const float4 *)p)[i];
                    ev[2 * i] = v.x; od[2 * i] = v.y; ev[2 * i + 1] = v.z; od[2 * i + 1] = v.w;
                }
            } else {
#pragma unroll
                for (int i = 0; i < 16; ++i) { ev[i] = p[2 * i]; od[i] = p[2 * i + 1]; }
            }
        }
        any |= gm_store_block(ev, od, o + ((size_t)t * nQ + (k >> 4)) * G6_QB, more,
                              gm_eight<true>(ev, od), (k >> 2) & 3, k & 3);
    }
    any = __syncthreads_or(any);
    if (threadIdx.x == 0) {
        wrow[t] = any;
        if (any) *wide = 1;
    }
}

typedef int g6_v8i __attribute__((ext_vector_type(8)));

/* acc += A (FP4, scale byte J of sa) x B (FP6 piece, scale byte P of sb) */
template <int J, int P>
__device__ __forceinline__ k3v4f g6_mma(uint4 a, uint32_t sa, gm_v6u b, uint32_t sb, k3v4f acc)
{
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
        (g6_v8i{(int)a.x, (int)a.y, (int)a.z, (int)a.w, 0, 0, 0, 0}),
        (g6_v8i{(int)b[0], (int)b[1], (int)b[2], (int)b[3], (int)b[4], (int)b[5], 0, 0}), acc, 4, 2,
        J, (int)sa, P, (int)sb);
}

/* A use of an accumulator here: the matrix instructions that make it stay before this point and
 * the LDS reads that follow in the source after it (the instructions have no memory order of
 * their own, and the compiler would move them all behind the last read) */
__device__ __forceinline__ void g6_pin(k3v4f &v) { asm volatile("" : "+v"(v)); }

/* The workgroup's tile: uniform across it except the lane and the wave. */
struct G6Tile {
    int p0, np, nb, lane, w, row0;       /* row0: first feature (mode 0) or output row */
    int nK;                              /* 128-column steps */
    const K3ExpertQ *q;                  /* the expert's matrices */
    uint32_t lds;
    uint8_t *ldsp;
};

/* row block b of the tile in matrix u (mode 0: 0 gate, 1 up); blocks outside the matrix read its
 * block 0 and are never stored */
template <int MODE>
__device__ __forceinline__ const uint8_t *g6_block(const K3kGemm6 &g, const G6Tile &t, int u, int b)
{
    const int row = t.row0 + 16 * b;
    const uint8_t *m = MODE == 0 ? (u ? t.q->p3 : t.q->p1) : t.q->p2;
    return m + (size_t)(row < g.rows ? row / 16 : 0) * ((size_t)((g.K + 511) / 512) * G6_QT);
}

/* A tile's steps past the nK first (W): the 128-column steps in which one of its columns has a block
 * of eight pieces, in LDS at G6_LIST; returns how many. Every wave looks through the columns
 * (lane l: column l) and finds the same. */
template <int MODE>
__device__ __forceinline__ int g6_again(const K3kGemm6 &g, const G6Tile &t)
{
    const int nQ = (g.K + 511) / 512, p = t.p0 + (t.lane < t.np ? t.lane : 0);
    const int row = MODE == 0 ? g.perm[p] / g.topk : p;
    const bool mine = t.lane < t.np && g.wrow[row];
    const uint8_t *q = g.b + g.more + (size_t)row * nQ * G6_QB + 1536;
    uint16_t *list = (uint16_t *)(t.ldsp + G6_LIST);
    int n = 0;
    /* two quads' loads at a time (a step's at a time: gate/up of 4,096 tokens with such blocks in
     * one of 50 3.06 instead of 3.01 ms) */
    for (int Q = 0; Q < nQ; Q += 2) {
        uint4 v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            v[i] = gm_ld16(q + (size_t)min(Q + (i >> 2), nQ - 1) * G6_QB + 16 * (i & 3));
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int c = 4 * Q + i;
            if (!__any(mine && (v[i].x | v[i].y | v[i].z | v[i].w)) || c >= t.nK) continue;
            if (threadIdx.x == 0) list[n] = (uint16_t)c;
            ++n;
        }
    }
    __syncthreads();
    return n;
}

/* One tile's products. The copies of a step: wave w takes column block w (NB = 3, 4), half a block
 * (NB = 2), or half of one's lines (NB = 1); lane 8 c + s of an instruction brings unit s ^ c
 * of its column's line to LDS unit 8 c + s. Weights are loaded DEPTH steps ahead. With 2 and 3
 * blocks the copies are issued two steps ahead as well (three stages): one step ahead, every
 * step lasted a trip to memory and then the matrix work (K3, 36 pairs an expert: 1.94 ms of
 * weights + 0.84 of matrix work took 2.80 ms; 2.56 so, and down 1.46 -> 1.36). With one block,
 * short steps, that is 2 % slower. Step c waits for all but the loads of step c + 1's weights;
 * of the three-stage order the wait takes in as many of those loads as there are copies behind
 * them, so the scales, three times of four already in the cache, are loaded first.
 * W: after the nK steps those of g6_again with the second array, a block without a place there as
 * zeros; the activations' scales are copied with every step. */
template <int MODE, int NB, int RG, bool W = false>
__device__ __forceinline__ void g6_run(const K3kGemm6 &g, const G6Tile &t)
{
    /* 128 accumulators leave room for the weights of one step ahead only */
    constexpr int DEPTH = RG * NB > 24 ? 1 : 2, NBUF = DEPTH + 1;
    constexpr int NST = DEPTH == 2 && NB > 1 && NB <= 3 ? 3 : 2;
    constexpr int STAGE = NB * G6_BLK, SCL0 = NST * STAGE, SCL = NB * 1024;
    static_assert(SCL0 + (W ? NST : 2) * SCL <= G6_LIST, "LDS");
    const int nS = W ? t.nK + g6_again<MODE>(g, t) : t.nK;
    /* step c's columns, and where its activations are */
    auto at = [&](int c) {
        return !W || c < t.nK ? c : gm_uniform(((const uint16_t *)(t.ldsp + G6_LIST))[c - t.nK]);
    };
    const int lane = t.lane, c16 = lane & 15, q4 = lane >> 4;
    k3v4f acc[RG][NB];
#pragma unroll
    for (int r = 0; r < RG; ++r)
#pragma unroll
        for (int n = 0; n < NB; ++n) acc[r][n] = k3v4f{0.f, 0.f, 0.f, 0.f};

    const int nQ = (g.K + 511) / 512;
    const int blk = NB >= 3 ? t.w : NB == 2 ? t.w >> 1 : 0;
    auto rowof = [&](int c) {            /* activation row of column c of the wave's block */
        const int col = 16 * blk + c;
        const int p = t.p0 + (col < t.np ? col : 0);
        const int row = MODE == 0 ? g.perm[p] / g.topk : p;
        return g.b + (size_t)row * nQ * G6_QB;
    };
    constexpr int NH = NB >= 3 ? 2 : 1;
    const int h0 = NB >= 3 ? 0 : t.w & 1;                    /* first half of the block */
    const int l0 = NB == 1 ? 2 * (t.w >> 1) : 0, l1 = NB == 1 ? (t.w < 2 ? 2 : 3) : 3;
    const bool does_scales = NB >= 3 || (NB == 2 ? (t.w & 1) == 0 : t.w == 2);
    const uint8_t *src[NH], *ssrc;
#pragma unroll
    for (int h = 0; h < NH; ++h)
        src[h] = rowof(8 * (h0 + h) + (lane >> 3)) + 16 * ((lane & 7) ^ (lane >> 3));
    ssrc = rowof(lane >> 2) + 1536 + 16 * (lane & 3);
    auto copy = [&](int s, int stage) {
        if (NB == 3 && t.w == 3) return;
        const int c = at(s);
        const size_t o = (size_t)(c >> 2) * G6_QB + (W && s >= t.nK ? g.more : 0);
        const uint32_t l = t.lds + stage * STAGE + blk * G6_BLK;
#pragma unroll
        for (int h = 0; h < NH; ++h)
#pragma unroll
            for (int n = 0; n < 3; ++n)
                if (NB > 1 || (n >= l0 && n < l1))
                    gm_dma16(src[h] + o + 384 * (c & 3) + 128 * n,
                             l + 1024 * (2 * n + h0 + h));
        if ((W || (c & 3) == 0) && does_scales)
            gm_dma16(ssrc + o, t.lds + SCL0 + (W ? stage : (c >> 2) & 1) * SCL + blk * 1024);
    };
    /* the wave's row blocks: mode 0 the gates' and then the ups' of its features */
    const uint8_t *rbase[RG];
#pragma unroll
    for (int r = 0; r < RG; ++r)
        rbase[r] = gm_uniform_ptr(
            MODE == 0 ? g6_block<MODE>(g, t, r < RG / 2 ? 0 : 1, RG / 2 * t.w + r % (RG / 2))
                      : g6_block<MODE>(g, t, 0, RG * t.w + r));
    uint4 wb[NBUF][RG];
    uint32_t ws[NBUF][RG];
    auto wload = [&](int k, uint4 (&d)[RG], uint32_t (&s)[RG]) {
        const int c = at(k);
        const size_t qo = (size_t)(c >> 2) * G6_QT;
#pragma unroll
        for (int r = 0; r < RG; ++r) s[r] = gm_ld4(rbase[r] + qo + 4096 + 4 * lane);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < RG; ++r) d[r] = gm_ld16(rbase[r] + qo + 1024 * (c & 3) + 16 * lane);
        __builtin_amdgcn_sched_barrier(0);
    };
    /* piece p of column c16's block q4: 16 bytes at bx (bx ^ 64 for odd p) in lines p / 2, 8
     * bytes at by ^ 32 p in line 2; its scales at bz */
    const uint32_t bx = (c16 >> 3) * 1024 + (c16 & 7) * 128 + 16 * (q4 ^ (c16 & 7));
    const uint32_t by = 4096 + (c16 >> 3) * 1024 + (c16 & 7) * 128 +
                        16 * ((q4 >> 1) ^ (c16 & 7)) + 8 * (q4 & 1);
    const uint32_t bz = SCL0 + 64 * c16 + 4 * q4;
    auto step = [&](int s, int stage, const uint4 (&w)[RG], const uint32_t (&sc)[RG], uint4 (&nw)[RG],
                    uint32_t (&ns)[RG]) {
        gm_wait_vm<(DEPTH == 2 ? 2 * RG : 0)>();
        __syncthreads();
        if (NST == 2 && s + 1 < nS) copy(s + 1, 1 - stage);
        wload(min(s + DEPTH, nS - 1), nw, ns);
        if (NST == 3 && s + 2 < nS) copy(s + 2, (stage + 2) % 3);
        __builtin_amdgcn_sched_barrier(0);
        if (s >= nS) return;
        const int c = at(s);
        const uint8_t *st = t.ldsp + stage * STAGE;
        const uint8_t *sl = t.ldsp + (W ? stage : (c >> 2) & 1) * SCL + 16 * (c & 3) + bz;
        const int sh = 8 * (c & 3);
        uint32_t sa[RG];
#pragma unroll
        for (int r = 0; r < RG; ++r) sa[r] = sc[r] >> sh;
        /* B operands two pieces ahead of their matrix instructions */
        gm_v6u b[3];
        uint32_t sb[2];
        auto bread = [&](int i) {
            const int n = i >> 2, p = i & 3;
            const uint4 u = *(const uint4 *)(st + (p & 1 ? bx ^ 64 : bx) + n * G6_BLK +
                                             2048 * (p >> 1));
            const uint2 v = *(const uint2 *)(st + (by ^ 32 * p) + n * G6_BLK);
            b[i % 3] = gm_v6u{u.x, u.y, u.z, u.w, v.x, v.y};
            if (p == 0) sb[n & 1] = *(const uint32_t *)(sl + 1024 * n);
            if (W && sb[n & 1] == 0) b[i % 3] = gm_v6u{};
        };
        bread(0);
        bread(1);
#pragma unroll
        for (int i = 0; i < 4 * NB; ++i) {
            const int n = i >> 2;
            if (i + 2 < 4 * NB) bread(i + 2);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < RG; ++r) {
                k3v4f &a = acc[r][n];
                if ((i & 3) == 0) a = g6_mma<0, 0>(w[r], sa[r], b[i % 3], sb[n & 1], a);
                if ((i & 3) == 1) a = g6_mma<0, 1>(w[r], sa[r], b[i % 3], sb[n & 1], a);
                if ((i & 3) == 2) a = g6_mma<0, 2>(w[r], sa[r], b[i % 3], sb[n & 1], a);
                if ((i & 3) == 3) a = g6_mma<0, 3>(w[r], sa[r], b[i % 3], sb[n & 1], a);
            }
#pragma unroll
            for (int r = 0; r < RG; ++r) g6_pin(acc[r][n]);
        }
    };
    if (NST == 2) copy(0, 0);
#pragma unroll
    for (int s = 0; s < DEPTH; ++s) {
        wload(min(s, nS - 1), wb[s], ws[s]);
        if (NST == 3 && s < nS) copy(s, s);
    }
    for (int c = 0; c < nS; c += NBUF) {
#pragma unroll
        for (int u = 0; u < NBUF; ++u)
            step(c + u, NST == 3 ? u : (c + u) & 1, wb[u], ws[u], wb[(u + DEPTH) % NBUF], ws[(u + DEPTH) % NBUF]);
    }
    gm_wait_vm<0>();

    if constexpr (MODE == 0) {
        __syncthreads();                 /* every wave is done with the LDS */
        gm_store_h<RG, NB>(acc, (float *)(t.ldsp + t.w * GM_HLDS), lane,
                           t.row0 + 8 * RG * t.w, g.rows, t.p0, t.np, g.b1, g.b2, g.h, g.hmore,
                           g.hrow, g.hwide);
    } else {
#pragma unroll
        for (int n = 0; n < NB; ++n) {
            const int col = 16 * n + c16;
            if (col < t.np) {
                const int row = t.row0 + 16 * RG * t.w;
                float *o = g.out + (size_t)g.perm[t.p0 + col] * g.ldo + row + 4 * q4;
#pragma unroll
                for (int r = 0; r < RG; ++r)
                    if (row + 16 * r < g.rows) *(k3v4f *)(o + 16 * r) = acc[r][n];
            }
        }
    }
}

/* The workgroup's tile: column tiles of more than 64 pairs are two of up to 64, one after the
 * other in an XCD's order, so that the second finds the weights in the XCD's L2. Returns 16 RG +
 * the column blocks, 0 for a workgroup without work. RG = 8 halves the activation copies, which
 * pays from 3 column blocks on (down at 1,024 and 4,096 tokens of the K2 layer: at 1 and 2
 * blocks 4 is 2-4 % faster, at 3 and 4 blocks 8 is by 5-10 %), once there are two rounds of
 * workgroups for every CU. Items with blocks of eight pieces: RG = 4, and 256 more. */
template <int MODE>
__device__ __forceinline__ int g6_setup(const K3kGemm6 &g, G6Tile &t, uint8_t *lds)
{
    const int ntl = *g.ntiles;
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const int rnd = slot / g.nft, ft = slot - rnd * g.nft;
    const int item = gm_item_of(rnd, xcd, ntl, !g.halves);
    if (item >= (ntl << g.halves)) return 0;
    const int4 tv = ((const int4 *)g.tiles)[item >> g.halves];
    const int e = gm_uniform(tv.x), hf = 64 * (item & g.halves);
    t.np = gm_uniform(tv.z) - hf;
    if (t.np <= 0) return 0;
    t.np = min(t.np, 64);
    t.p0 = gm_uniform(tv.y) + hf;
    t.nb = (t.np + 15) >> 4;
    t.lane = threadIdx.x & 63;
    t.w = gm_uniform(threadIdx.x >> 6);
    t.nK = (g.K + 127) / 128;
    bool wide = false;
    if (*g.wide) {
        const int p = t.p0 + min(t.lane, t.np - 1);
        wide = __any(g.wrow[MODE == 0 ? g.perm[p] / g.topk : p] != 0);
    }
    const bool big = !wide && t.nb >= 3 && ntl * ((g.nft + 1) / 2) >= G6_BIG_MIN;
    if (big && 2 * ft >= g.nft) return 0;
    t.row0 = (MODE == 0 ? G6_ROWS / 2 : G6_ROWS) * ft * (big ? 2 : 1);
    t.ldsp = lds;
    t.lds = (uint32_t)(uintptr_t)(k3lds)lds;
    t.q = g.eq + e;
    return (wide ? 256 : 0) + 16 * (big ? 8 : 4) + t.nb;
}
