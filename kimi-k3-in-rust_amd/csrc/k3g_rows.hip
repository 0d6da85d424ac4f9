/* k3g_rows.hip - the routed experts of checkpoint-layout (row-major) MXFP4 weights on the scaled
 * FP4 x FP6 matrix instructions.
 *
 * The engine computes, per (token, slot) pair, three MXFP4 GEMVs per expert
 * (src/core/k3_ops.c:604-640, :751-778); here an expert's pairs share one pass over its rows,
 * eight at a time. The codes and scales go to v_mfma_scale_f32_16x16x128_f8f6f4 as they are
 * stored. An activation is the sum of eight FP6 (E2M3) pieces, each with its own E8M0 scale per
 * 32 values: each piece leaves at most 1/16 of the block's largest value and 1/32 in the mean,
 * so eight hold fp32's 24 bits of values down to 2^-8 of the largest at worst, 2^-16 in the mean
 * (beside one 10^6 times as large 1.6e-8 is left of normally distributed values, 2-norm). A pair
 * with a block where that is not enough is summed without pieces (k_rows_x). The pieces are eight
 * columns of the B operand (two pairs per instruction, columns 8 pi + piece), 128 products
 * sum exactly before they are added to the fp32 accumulator, and a row's result is the
 * sum of its eight columns.
 *
 * Bound by the weight stream. A wave's operand rows are 64 bytes at a stride of a whole row, which
 * the cache serves badly (each line is asked for in two halves), so every wave copies its own
 * 32 rows through LDS, eight rows x one 128-byte line per global_load_lds_dwordx4, 256 columns
 * two intervals ahead, in units swizzled by the row so that the operand reads meet no bank
 * conflict; the rows' scale bytes follow per 512 columns, as the aligned words that hold them.
 * Two workgroups of 4 waves per CU keep 64 KB of weights in flight. Measured, 28 experts of 4
 * tokens (7168 x 2048, 655 MB): gate/up 753 -> 95 us (4.6 TB/s), down 441 -> 62 us (3.5 TB/s)
 * against a wave per row tile with fp32 multiply-adds, which decodes every weight once per
 * four tokens; error against 64 bits 3.2e-7 -> 1.6e-7.
 *
 * Activation rows: per 128 columns 800 bytes: dwords 0 .. 3 of piece p of block q at
 * 16 (4 p + q), dwords 4 and 5 at 512 + 8 (4 p + q), the scale byte at 768 + 4 p + q; a row is
 * whole intervals of 256 columns, zero past the end. */
#include "k3g_gemm.h"

#define RW_STEP 800                 /* bytes of 128 columns of an activation row */
#define RW_NP 8                     /* pieces */
#define RW_PAIRS 8                  /* pairs per pass */
#define RW_WST 4096                 /* a wave's weights of one interval: 32 rows x 128 bytes */
#define RW_SCL 768                  /* a wave's scales of two intervals: 32 rows x 20 bytes */
#define RW_BST ((RW_PAIRS * 2 * RW_STEP + 1023) / 1024 * 1024)   /* whole copy instructions */
#define RW_B0 (4 * 3 * RW_WST)
#define RW_S0 (RW_B0 + 2 * RW_BST)
#define RW_LDS (RW_S0 + 4 * 2 * RW_SCL)

typedef int rw_v8i __attribute__((ext_vector_type(8)));

/* x (fp32 [T][K]) -> activation rows, one thread per block of 32. The scales are NaN where a value
 * is not finite, and where the pieces leave more than 2^-22 of all but one or an eighth of the
 * block's values that are not zero: values of less than about 2^-20 of its largest, or a block that
 * small that a scale has no byte. The row's products are then NaN, and are summed again from the
 * fp32 values (rw_plain). */
__global__ void __launch_bounds__(256)
k_rows_x(const float *__restrict__ x, int T, int K, uint8_t *__restrict__ o)
{
    const int nbk = 8 * ((K + 255) / 256);
    const long long b = (long long)blockIdx.x * 256 + threadIdx.x;
    if (b >= (long long)T * nbk) return;
    const int t = (int)(b / nbk), k = (int)(b - (long long)t * nbk);
    gm_v16f ev = {}, od = {};
    if (32 * k < K) {
        const float4 *src = (const float4 *)(x + (size_t)t * K + 32 * k);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float4 v = src[i];
            ev[2 * i] = v.x; od[2 * i] = v.y; ev[2 * i + 1] = v.z; od[2 * i + 1] = v.w;
        }
    }
    const gm_v16f ev0 = ev, od0 = od;
    uint32_t d[6 * RW_NP];
    uint8_t s[RW_NP];
    gm_pieces<RW_NP>(ev, od, d, s);
    constexpr int LP = 6 * (RW_NP - 1);
    gm_less(ev, od, gm_v6u{d[LP], d[LP + 1], d[LP + 2], d[LP + 3], d[LP + 4], d[LP + 5]}, s[RW_NP - 1]);
    int n = 0, left = 0;
    auto look = [&](float v, float r) {
        n += v != 0.0f;
        left += fabsf(r) > 0x1p-22f * fabsf(v);
    };
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        look(ev0[i], ev[i]);
        look(od0[i], od[i]);
    }
    const bool bad = gm_bad(ev0, od0) || (left > 0 && left >= n - 1 - n / 8);
    uint8_t *q = o + ((size_t)t * (nbk / 4) + (k >> 2)) * RW_STEP;
#pragma unroll
    for (int p = 0; p < RW_NP; ++p) {
        const int u = 4 * p + (k & 3);
        *(uint4 *)(q + 16 * u) = make_uint4(d[6 * p], d[6 * p + 1], d[6 * p + 2], d[6 * p + 3]);
        *(uint2 *)(q + 512 + 8 * u) = make_uint2(d[6 * p + 4], d[6 * p + 5]);
        q[768 + u] = bad ? 255 : s[p];
    }
}

/* A row's product column by column: what an infinity or NaN, a sum that overflowed, or a block of
 * too wide a range needs, for the pieces have no infinities. One lane sums all columns, so in
 * double. */
__device__ __attribute__((noinline)) float rw_plain(const uint8_t *w, const uint8_t *s,
                                                    const float *x, int K)
{
    double a = 0.0;
    for (int c = 0; c < K; c += 8) {
        uint32_t v;
        __builtin_memcpy(&v, w + c / 2, 4);
        float f[8];
        k3d_fp4x8(v, k3d_e8m0(s[c / 32]), f);
#pragma unroll
        for (int i = 0; i < 8; ++i) a = fma((double)f[i], (double)x[c + i], a);
    }
    return (float)a;
}

/* One pass over a workgroup's rows for the np <= 2 NG pairs at sorted positions p0 .. */
template <int MODE, int NG>
__device__ __forceinline__ void rw_pass(const K3kRows &g, const K3ExpertQ &q, int row0, int p0,
                                        int np, uint8_t *ldsp, uint32_t lds)
{
    const int lane = threadIdx.x & 63, w = gm_uniform(threadIdx.x >> 6);
    const int c16 = lane & 15, q4 = lane >> 4;
    const int kb = g.K / 2, ks = g.K / 32;               /* bytes of a row's codes, of its scales */
    const int nS = (g.K + 255) / 256;                    /* intervals */
    const int ns = 2 * nS;
    k3v4f acc[2][NG];
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int n = 0; n < NG; ++n) acc[r][n] = k3v4f{0.f, 0.f, 0.f, 0.f};

    /* the wave's row i < 32: mode 0: gate row i, then up row i - 16, of its 16 features; mode 1:
     * its 32 output rows. Rows past the matrix read its last one and are never stored. */
    auto row = [&](int i) { return min(row0 + (MODE == 0 ? 16 * w + (i & 15) : 32 * w + i), g.rows - 1); };
    auto mat = [&](int i) { return MODE == 0 ? (i < 16 ? q.p1 : q.p3) : q.p2; };
    auto smat = [&](int i) { return MODE == 0 ? (i < 16 ? q.s1 : q.s3) : q.s2; };
    const uint8_t *wsrc[4];
    const int unit = 16 * ((lane & 7) ^ (lane >> 3));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 8 * i + (lane >> 3);
        wsrc[i] = mat(8 * i) + (size_t)row(r) * kb;
    }
    /* the copy instruction takes whole aligned units; other rows pass through registers */
    const bool whole = (((MODE == 0 ? (uintptr_t)q.p1 | (uintptr_t)q.p3 : (uintptr_t)q.p2)) & 15) == 0;
    /* the words that hold the scale bytes 16 Q .. 16 Q + 15 of a row: word (lane, i) is word d of
     * row r, 4 d - mis bytes into the 16 */
    const uint8_t *ssrc[3];
    int smax[3], sd[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int u = min(64 * i + lane, 159), r = u / 5;
        const uint8_t *p = smat(r) + (size_t)row(r) * ks;
        const int mis = (int)((uintptr_t)p & 3);
        ssrc[i] = p - mis;
        sd[i] = u - 5 * r;
        smax[i] = (mis + ks - 1) >> 2;                   /* the row's last word */
    }
    uint32_t sat[2];                                     /* where this lane's scales start */
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const int i = 16 * r + c16;
        const int mis = (int)((uintptr_t)(smat(i) + (size_t)row(i) * ks) & 3);
        sat[r] = (uint32_t)(RW_S0 + w * 2 * RW_SCL + 20 * i + mis + q4);
    }
    /* the activation copies: 200 NG units of 16 bytes an interval, wave w the 64-unit instructions
     * w, w + 4, ... */
    constexpr int UP = RW_STEP / 8, NI = (2 * UP * NG + 63) / 64, NB = (NI + 3) / 4;
    const uint8_t *bsrc[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const int u = min(64 * (4 * i + w) + lane, 2 * UP * NG - 1), pi = u / UP;
        const int p = g.perm[p0 + (pi < np ? pi : 0)];
        bsrc[i] = g.x + (size_t)(MODE == 0 ? p / g.topk : p) * ns * RW_STEP + 16 * (u - UP * pi);
    }
    auto bcopy = [&](int s) {
        const uint32_t l = lds + RW_B0 + (s & 1) * RW_BST;
#pragma unroll
        for (int i = 0; i < NB; ++i)
            if (4 * i + w < NI)
                gm_dma16(bsrc[i] + (size_t)min(s, nS - 1) * 2 * RW_STEP, l + 1024 * (4 * i + w));
    };
    auto wcopy = [&](int s, int slot) {
        const int o = min(128 * min(s, nS - 1) + unit, kb - 16);
        const uint32_t l = (3 * w + slot) * RW_WST;
        if (whole) {
#pragma unroll
            for (int i = 0; i < 4; ++i) gm_dma16(wsrc[i] + o, lds + l + 1024 * i);
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint8_t *p = wsrc[i] + o;
                *(uint4 *)(ldsp + l + 1024 * i + 16 * lane) =
                    make_uint4(gm_ld4(p), gm_ld4(p + 4), gm_ld4(p + 8), gm_ld4(p + 12));
            }
        }
        if (!(s & 1)) {
            const int Q = min(s, nS - 1) >> 1;
            const uint32_t sl = lds + RW_S0 + (2 * w + ((s >> 1) & 1)) * RW_SCL;
#pragma unroll
            for (int i = 0; i < 3; ++i)
                gm_dma4(ssrc[i] + 4 * min(4 * Q + sd[i], smax[i]), sl + 256 * i);
        }
    };
    /* operand reads: row i's unit u of an interval at (i / 8) 1024 + (i % 8) 128 + 16 (u ^ i % 8);
     * column 8 pi + piece */
    const uint32_t abase = 3 * w * RW_WST + (c16 >> 3) * 1024 + (c16 & 7) * 128;
    const int bu = 4 * (c16 & 7) + q4;
    const uint32_t bbase = RW_B0 + (c16 >> 3) * 2 * RW_STEP;
    auto interval = [&](auto par, int s, int slot) {
        constexpr int PAR = decltype(par)::value;
        /* all but the copies of interval s + 1's weights (and, with an even one, its scales) */
        gm_wait_vm<(PAR == 0 ? 4 : 7)>();
        __syncthreads();
        bcopy(s + 1);
        wcopy(s + 2, slot == 0 ? 2 : slot - 1);
        const uint32_t so = ((s >> 1) & 1) * RW_SCL + 8 * PAR;
#pragma unroll
        for (int st = 0; st < 2; ++st) {
            if (256 * s + 128 * st >= g.K) break;
            uint4 a[2];
            uint32_t sa[2];
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                a[r] = *(const uint4 *)(ldsp + abase + slot * RW_WST + 2048 * r +
                                        16 * ((4 * st + q4) ^ (c16 & 7)));
                sa[r] = ldsp[sat[r] + so + 4 * st];
                /* blocks past the row meet zero activations: any finite scale; the byte 255 is a
                 * block of zeros (src/core/k3_ops.c:1315-1322) */
                const bool out = 8 * s + 4 * st + q4 >= ks;
                if (sa[r] == 255 || out) {
                    a[r] = make_uint4(0, 0, 0, 0);
                    sa[r] = 127;
                }
            }
#pragma unroll
            for (int n = 0; n < NG; ++n) {
                const uint8_t *b = ldsp + bbase + (s & 1) * RW_BST + (4 * n + st) * RW_STEP;
                const uint4 u = *(const uint4 *)(b + 16 * bu);
                const uint2 v = *(const uint2 *)(b + 512 + 8 * bu);
                const int sb = b[768 + bu];
#pragma unroll
                for (int r = 0; r < 2; ++r)
                    acc[r][n] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                        (rw_v8i{(int)a[r].x, (int)a[r].y, (int)a[r].z, (int)a[r].w, 0, 0, 0, 0}),
                        (rw_v8i{(int)u.x, (int)u.y, (int)u.z, (int)u.w, (int)v.x, (int)v.y, 0, 0}),
                        acc[r][n], 4, 2, 0, (int)sa[r], 0, sb);
            }
        }
    };
    /* the first interval's and the second's weights, in the order of the loop */
    wcopy(0, 0);
    bcopy(0);
    wcopy(1, 1);
    int slot = 0;
    for (int s = 0; s < nS; s += 2) {
        interval(GmInt<0>{}, s, slot);
        slot = slot == 2 ? 0 : slot + 1;
        if (s + 1 < nS) {
            interval(GmInt<1>{}, s + 1, slot);
            slot = slot == 2 ? 0 : slot + 1;
        }
    }
    gm_wait_vm<0>();
    __syncthreads();                     /* the next pass copies into the same LDS */

    /* the columns of a pair summed; lane piece i < 4 of the eight finishes element i */
#pragma unroll
    for (int n = 0; n < NG; ++n) {
        const int pi = 2 * n + (c16 >> 3), e = c16 & 7;
        float v[2];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            k3v4f t = acc[r][n];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float x = t[i];
                x += __shfl_xor(x, 4, K3G_WAVE);
                x += __shfl_xor(x, 2, K3G_WAVE);
                x += __shfl_xor(x, 1, K3G_WAVE);
                t[i] = x;
            }
            v[r] = e == 0 ? t[0] : e == 1 ? t[1] : e == 2 ? t[2] : t[3];
        }
        if (e < 4 && pi < np) {
            const int p = g.perm[p0 + pi];
            const float *x = g.z + (size_t)(MODE == 0 ? p / g.topk : p) * g.K;
#pragma unroll
            for (int r = 0; r < 2; ++r)
                if (!(fabsf(v[r]) < __builtin_inff())) {
                    const int i = 16 * r + 4 * q4 + e;
                    v[r] = rw_plain(mat(i) + (size_t)row(i) * kb, smat(i) + (size_t)row(i) * ks, x,
                                    g.K);
                }
            if (MODE == 0) {
                const int f = row0 + 16 * w + 4 * q4 + e;
                if (f < g.rows) g.h[(size_t)p * g.rows + f] = k3d_act(v[0], v[1], g.b1, g.b2);
            } else {
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    const int o = row0 + 32 * w + 16 * r + 4 * q4 + e;
                    if (o < g.rows) g.out[(size_t)p * g.rows + o] = v[r];
                }
            }
        }
    }
}

/* grid (row tiles, active experts bound): 64 features (mode 0) or 128 output rows (mode 1) of
 * one active expert, its pairs eight at a time */
template <int MODE>
__global__ void __launch_bounds__(256, 2)
k_rows(const K3kRows g)
{
    __shared__ __attribute__((aligned(1024))) uint8_t lds[RW_LDS];
    static_assert(2 * RW_LDS <= 160 * 1024, "two workgroups per CU");
    if ((int)blockIdx.y >= *g.nact) return;
    const int e = gm_uniform(g.act[blockIdx.y]);
    const K3ExpertQ q = g.eq[e];
    const int row0 = (MODE == 0 ? 64 : 128) * blockIdx.x;
    const int beg = gm_uniform(g.off[e]), end = gm_uniform(g.off[e + 1]);
    const uint32_t l = (uint32_t)(uintptr_t)(k3lds)lds;
    for (int p0 = beg; p0 < end; p0 += RW_PAIRS) {
        const int np = min(end - p0, RW_PAIRS);
        if (np <= 2) rw_pass<MODE, 1>(g, q, row0, p0, np, lds, l);
        else if (np <= 4) rw_pass<MODE, 2>(g, q, row0, p0, np, lds, l);
        else rw_pass<MODE, 4>(g, q, row0, p0, np, lds, l);
    }
}

extern "C" size_t k3k_rows_bytes(int K) { return (size_t)((K + 255) / 256) * 2 * RW_STEP; }

extern "C" int k3k_rows_x(const float *x, int T, int K, uint8_t *o, hipStream_t st)
{
    if (T < 1 || K < 32 || K % 32 || (((uintptr_t)x | (uintptr_t)o) & 15)) return -1;
    const long long n = (long long)T * 8 * ((K + 255) / 256);
    hipLaunchKernelGGL(k_rows_x, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, x, T, K, o);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" int k3k_rows(const K3kRows *g, int maxU, hipStream_t st)
{
    if (g->mode < 0 || g->mode > 1 || !g->eq || !g->z || !g->x || ((uintptr_t)g->x & 15) || !g->act ||
        !g->nact || !g->off || !g->perm || g->topk < 1 || g->K < 32 || g->K % 32 || g->rows < 1 ||
        maxU < 1 || (g->mode == 0 ? !g->h : !g->out))
        return -1;
    const int per = g->mode == 0 ? 64 : 128;
    const dim3 grid((unsigned)((g->rows + per - 1) / per), (unsigned)maxU);
    if (g->mode == 0) hipLaunchKernelGGL(k_rows<0>, grid, dim3(256), 0, st, *g);
    else hipLaunchKernelGGL(k_rows<1>, grid, dim3(256), 0, st, *g);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
