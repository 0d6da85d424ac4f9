/* k3g_gemm.h - device helpers of the grouped GEMMs (k3g_gemm.hip, k3g_gemm6.h). */
#pragma once

#include "k3g_dev.h"
#include "k3g_kernels.h"

typedef float k3v4f __attribute__((ext_vector_type(4)));
typedef __bf16 k3v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 k3v2bf __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void *k3lds;

__device__ __forceinline__ int gm_uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

/* Loads through pointers the compiler cannot prove global (they come from the expert
 * table) would be flat loads, which also count against the LDS counter and make every
 * ds_read wait for outstanding HBM loads: address them as global memory explicitly. */
typedef unsigned int gm_v4u __attribute__((ext_vector_type(4)));
typedef unsigned int gm_v2u __attribute__((ext_vector_type(2)));
#ifdef __HIP_DEVICE_COMPILE__
typedef const __attribute__((address_space(1))) gm_v4u *gm_g4;
typedef const __attribute__((address_space(1))) gm_v2u *gm_g2;
typedef const __attribute__((address_space(1))) uint32_t *gm_g1;
#else
typedef const gm_v4u *gm_g4;       /* the host pass only parses device code */
typedef const gm_v2u *gm_g2;
typedef const uint32_t *gm_g1;
#endif

__device__ __forceinline__ uint4 gm_ld16(const void *p)
{
    const gm_v4u v = *(gm_g4)p;
    return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ uint32_t gm_ld4(const void *p) { return *(gm_g1)p; }

/* One DMA instruction: 64 lanes x 16 bytes from their own global addresses to 1 KB of LDS
 * at byte address `lds` (lane l at lds + 16 l). Issued as inline assembly so the
 * compiler does not treat every later LDS read as waiting on it (it would drain all
 * outstanding loads before each ds_read); completion is awaited explicitly with
 * s_waitcnt vmcnt before the barrier that publishes the stage. M0 is saved and restored
 * around the instruction, which needs one wait state after M0 is written. */
__device__ __forceinline__ void gm_dma16(const void *src, uint32_t lds)
{
    uint32_t keep;
    asm volatile("s_mov_b32 %0, m0\n\t"
                 "s_mov_b32 m0, %2\n\ts_nop 0\n\t"
                 "global_load_lds_dwordx4 %1, off\n\t"
                 "s_mov_b32 m0, %0"
                 : "=&s"(keep) : "v"(src), "s"(lds) : "memory");
}

/* 64 lanes x 4 bytes, lane l at lds + 4 l */
__device__ __forceinline__ void gm_dma4(const void *src, uint32_t lds)
{
    uint32_t keep;
    asm volatile("s_mov_b32 %0, m0\n\t"
                 "s_mov_b32 m0, %2\n\ts_nop 0\n\t"
                 "global_load_lds_dword %1, off\n\t"
                 "s_mov_b32 m0, %0"
                 : "=&s"(keep) : "v"(src), "s"(lds) : "memory");
}

/* a wave-uniform pointer, in scalar registers */
template <typename P>
__device__ __forceinline__ P *gm_uniform_ptr(P *p)
{
    const uint64_t v = (uint64_t)(uintptr_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (P *)(uintptr_t)(((uint64_t)hi << 32) | lo);
}

/* s_waitcnt vmcnt(N) (expcnt, lgkmcnt not waited on) */
template <int N>
__device__ __forceinline__ void gm_wait_vm()
{
    static_assert(N >= 0 && N < 64, "vmcnt");
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | (N >> 4) << 14);
}

/* Workgroup b of a grouped launch runs on XCD b % 8 and is dispatched there in the order of
 * b / 8: round r of XCD x. The column tiles (largest first) are dealt to the XCDs in groups of
 * G = K3G_TILE_GROUP consecutive tiles, the groups in a snake: round r of XCD x takes tile
 * G (8 q + x) + r % G (q = r / G even) or G (8 q + 7 - x) + r % G (q odd), so every XCD gets
 * the same mix, largest first, and an expert's consecutive full tiles land on one XCD in
 * consecutive rounds. */
__device__ __forceinline__ int gm_tile_of(int rnd, int xcd)
{
    const int grp = rnd / K3G_TILE_GROUP, gi = rnd - grp * K3G_TILE_GROUP;
    return K3G_TILE_GROUP * (8 * grp + ((grp & 1) ? 7 - xcd : xcd)) + gi;
}

/* The item of a round of n: as gm_tile_of; but where an expert is one item (single: as a
 * rule no two share weights) and the groups of four would leave the fullest XCD a sixth above the mean, one by
 * one. 40 items (5 tokens of the K2 layer) in groups are 8 for two XCDs and 4 for the others. Whole
 * calls, us: K2 at 5 / 6 / 10 / 16 tokens 287 / 307 / 427 / 561 -> 269 / 294 / 403 / 545, K3 at 5 /
 * 9 tokens 437 / 594 -> 417 / 580. */
__device__ __forceinline__ int gm_item_of(int rnd, int xcd, int n, bool single)
{
    if (!single || 7 * n > 6 * 8 * K3G_TILE_ROUNDS(n)) return gm_tile_of(rnd, xcd);
    return 8 * rnd + ((rnd & 1) ? 7 - xcd : xcd);
}

/* a compile-time integer as an argument */
template <int N> struct GmInt { static constexpr int value = N; };

/* Instrumentation: a workgroup's start and end as the records of its column tile and its `tall`
 * feature tiles of the nft, at their places in a launch of one item per column tile and one feature
 * tile per workgroup (the second half of a tile that is two items has none, nor do tiles from
 * `limit` on); every step-th feature tile has one. */
__device__ __forceinline__ void gm_trace(unsigned long long *trace, int nft, int step, int tall,
                                         int halves, int n, bool single, int limit,
                                         unsigned long long t_start)
{
    const int slot = blockIdx.x >> 3;
    const int rnd = slot / nft, f0 = tall * (slot - rnd * nft), nf = (nft + step - 1) / step;
    const int item = gm_item_of(rnd, blockIdx.x & 7, n, single), tile = item >> halves;
    if ((item & halves) || tile >= limit) return;
    const int grp = tile / K3G_TILE_GROUP, q = grp >> 3;
    const int xcd = (q & 1) ? 7 - (grp & 7) : grp & 7;
    const size_t r = (size_t)(K3G_TILE_GROUP * q + tile % K3G_TILE_GROUP) * nf;
    const unsigned long long t_end = wall_clock64();
    const unsigned long long id = (unsigned long long)(__builtin_amdgcn_s_getreg((3 << 11) | 20) & 15) << 32 |
                                  (unsigned)__builtin_amdgcn_s_getreg((31 << 11) | 4);
    for (int f = f0; f < min(f0 + tall, nft); ++f) {
        if (f % step) continue;
        unsigned long long *o = trace + 4 * (8 * (r + f / step) + xcd);
        o[0] = t_start;
        o[1] = t_end;
        o[2] = (unsigned long long)tile << 32 | (unsigned)(f / step);
        o[3] = id;
    }
}

typedef float gm_v16f __attribute__((ext_vector_type(16)));
typedef float gm_v32f __attribute__((ext_vector_type(32)));
typedef unsigned gm_v6u __attribute__((ext_vector_type(6)));

/* 32 floats (even and odd elements apart) / 2^(byte - 127) as E2M3, nearest-even, clamped to
 * +-7.5, element i in 6-bit field i; and back. Written as assembly for the early clobber: the
 * instruction writes its result while it still reads its sources, and the compiler's builtin
 * may give them the same registers. */
__device__ __forceinline__ gm_v6u gm_to_fp6(const gm_v16f &ev, const gm_v16f &od, float scale)
{
    gm_v6u r;
    asm("v_cvt_scalef32_2xpk16_fp6_f32 %0, %1, %2, %3" : "=&v"(r) : "v"(ev), "v"(od), "v"(scale));
    return r;
}

__device__ __forceinline__ gm_v32f gm_from_fp6(const gm_v6u &p, float scale)
{
    gm_v32f r;
    asm("v_cvt_scalef32_pk32_f32_fp6 %0, %1, %2" : "=&v"(r) : "v"(p), "v"(scale));
    return r;
}

/* ev, od less the piece w at its scale byte */
__device__ __forceinline__ void gm_less(gm_v16f &ev, gm_v16f &od, const gm_v6u &w, uint32_t sb)
{
    const gm_v32f y = gm_from_fp6(w, __uint_as_float(sb << 23));
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        ev[i] -= y[2 * i];
        od[i] -= y[2 * i + 1];
    }
}

/* 32 values (even and odd elements apart) as NP pieces: piece p's six dwords at d + 6 p, its E8M0
 * byte s[p]; each piece's scale puts the largest remainder in [4, 8), so a piece leaves at most
 * 1/16 of the block's largest remainder and 1/32 in the mean. ev and od become what the pieces
 * before the last leave. */
template <int NP>
__device__ __forceinline__ void gm_pieces(gm_v16f &ev, gm_v16f &od, uint32_t (&d)[6 * NP],
                                          uint8_t (&s)[NP])
{
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        float m = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) m = fmaxf(m, fmaxf(fabsf(ev[i]), fabsf(od[i])));
        const int sb = m > 0.0f ? max((int)(__float_as_uint(m) >> 23) - 2, 1) : 127;
        const gm_v6u w = gm_to_fp6(ev, od, __uint_as_float((uint32_t)sb << 23));
        if (p < NP - 1) gm_less(ev, od, w, sb);
#pragma unroll
        for (int i = 0; i < 6; ++i) d[6 * p + i] = w[i];
        s[p] = (uint8_t)sb;
    }
}

/* a value is infinite or NaN (pieces then mean nothing) */
__device__ __forceinline__ bool gm_bad(const gm_v16f &ev, const gm_v16f &od)
{
    bool bad = false;
#pragma unroll
    for (int i = 0; i < 16; ++i)
        bad |= !(fabsf(ev[i]) < __builtin_inff()) || !(fabsf(od[i]) < __builtin_inff());
    return bad;
}

/* Blocks that take eight pieces. Four leave 3e-7 of the block's largest value on every one of its
 * values; four more 2e-14 beside a value 16 times as large, 1.6e-11 beside 1000, 1.6e-8 beside
 * 10^6. The rules count the values of 1/8, 1/32 and 1/128 of the largest or more.
 *
 * x had been two bf16 pieces, 2.5e-6 of each value: less than four FP6 pieces leave below an eighth
 * of the largest. Eight where a few values (one and an eighth of those that are not zero) are that
 * large, or half are 1/32 or three quarters 1/128. What is left then of normally distributed values
 * beside 1, 4, 8 or 16 that are 16 times as large is 1.5e-6, 1.5e-6, 5e-6 and 9e-6 of them, beside
 * 100 times as large 7e-7, 6e-8, 0 and 0; and no block of 800,000 normally distributed ones takes
 * eight. (By the sum of the squared orders below the largest, which leaves more beside
 * outliers, 4 in a million did, so one in a dozen of full tiles: gate/up of 4,096 fp32 tokens 2.41
 * ms; four pieces everywhere 2.32, these rules within 1 % of that.)
 *
 * h had been a bf16 piece with an MXFP8 remainder, 3.9e-5 of each value: less than four FP6 pieces
 * leave below 1/130 of the largest. Where gates are large, half of the values of every block lie that
 * far below the other half (silu of a negative gate), and the block's products are those of the
 * larger half: eight only where few values are that large. (With the half as well, the down product
 * of 4,096 tokens of such a layer took nearly every step twice, 1.58 against 1.33 ms.) */
template <bool X>
__device__ __forceinline__ bool gm_eight(const gm_v16f &ev, const gm_v16f &od)
{
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) m = fmaxf(m, fmaxf(fabsf(ev[i]), fabsf(od[i])));
    int n = 0, c3 = 0, c5 = 0, c7 = 0;
    auto count = [&](float v) {
        v = fabsf(v);
        n += v != 0.0f;
        if (X) {
            c3 += v >= m * 0x1p-3f;
            c5 += v >= m * 0x1p-5f;
        }
        c7 += v >= m * 0x1p-7f;
    };
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        count(ev[i]);
        count(od[i]);
    }
    const int few = X ? c3 : c7;
    return (few <= 1 + n / 8 && few < n) || (X && (2 * c5 <= n || 4 * c7 <= 3 * n));
}

/* One block's four pieces in a quad (k3g_gemm6.h): step j, block q. */
__device__ __forceinline__ void gm_put_pieces(const uint32_t (&d)[24], uint32_t scales,
                                              uint8_t *quad, int j, int q)
{
    uint8_t *o = quad + 384 * j;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        *(uint4 *)(o + 64 * p + 16 * q) =
            make_uint4(d[6 * p], d[6 * p + 1], d[6 * p + 2], d[6 * p + 3]);
        *(uint2 *)(o + 256 + 32 * p + 8 * q) = make_uint2(d[6 * p + 4], d[6 * p + 5]);
    }
    *(uint32_t *)(quad + 1536 + 16 * j + 4 * q) = scales;
}

__device__ __forceinline__ uint32_t gm_bytes(const uint8_t (&s)[4])
{
    return s[0] | (uint32_t)s[1] << 8 | (uint32_t)s[2] << 16 | (uint32_t)s[3] << 24;
}

/* One block of 32 values into its place in a quad and, for a block of eight pieces (true if it is
 * stored as one), the next four into the same place `more` bytes on; elsewhere that place gets
 * scales of zero. A block with an infinity or NaN gets the NaN scale, so the products are NaN as
 * they were. */
__device__ __forceinline__ bool gm_store_block(gm_v16f ev, gm_v16f od, uint8_t *quad, size_t more,
                                               bool eight, int j, int q)
{
    uint32_t d[24];
    uint8_t s[4];
    const bool bad = gm_bad(ev, od), w = !bad && eight;
    gm_pieces<4>(ev, od, d, s);
    gm_put_pieces(d, bad ? 0xffffffffu : gm_bytes(s), quad, j, q);
    if (w) {
        gm_less(ev, od, gm_v6u{d[18], d[19], d[20], d[21], d[22], d[23]}, s[3]);
        gm_pieces<4>(ev, od, d, s);
        gm_put_pieces(d, gm_bytes(s), quad + more, j, q);
    } else {
        *(uint32_t *)(quad + more + 1536 + 16 * j + 4 * q) = 0;
    }
    return w;
}

/* This wave's LDS writes are visible to its own later reads, whichever lane made them */
__device__ __forceinline__ void gm_wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

/* bytes of LDS per wave that gm_store_h takes */
#define GM_HLDS 18432

/* A wave's gate and up sums (row groups r < RG / 2 the gates, the others the ups of the same 8 RG
 * features from f0 on; column block n's column lane % 16) -> activations -> h rows p0 + column
 * as FP6 quads of `rows` features (those past it zero; rows with blocks of eight pieces are marked in
 * wrow and raise *wide), columns below np. wl: GM_HLDS bytes of
 * LDS of this wave's own. The sums go to rows [feature block b][column block n][column c] of 32
 * gates and 32 ups (each padded to 36), the activations over the gates, eight per lane and
 * block; then every lane makes the pieces of one row. */
template <int RG, int NBW>
__device__ __forceinline__ void gm_store_h(k3v4f (&acc)[RG][NBW], float *wl, int lane, int f0,
                                           int rows, int p0, int np, float b1, float b2, uint8_t *h,
                                           size_t more, uint8_t *wrow, int32_t *wide)
{
    const int c16 = lane & 15, q4 = lane >> 4;
    const int nQh = (rows + 511) / 512;
    auto finish = [&](auto nc, auto cc) {
        constexpr int N0 = decltype(nc)::value, NN = decltype(cc)::value;
#pragma unroll
        for (int b = 0; b < RG / 4; ++b)
#pragma unroll
            for (int n = 0; n < NN; ++n) {
                float *o = wl + (16 * (b * NN + n) + c16) * 72 + 4 * q4;
                *(k3v4f *)o = acc[2 * b][N0 + n];
                *(k3v4f *)(o + 16) = acc[2 * b + 1][N0 + n];
                *(k3v4f *)(o + 36) = acc[RG / 2 + 2 * b][N0 + n];
                *(k3v4f *)(o + 52) = acc[RG / 2 + 2 * b + 1][N0 + n];
            }
        gm_wave_sync();
#pragma unroll 1
        for (int i = 0; i < RG / 2 * NN; ++i) {
            float *o = wl + (16 * (i >> 1) + c16) * 72 + 8 * q4 + 4 * (i & 1);
            const float4 gv = *(const float4 *)o, uv = *(const float4 *)(o + 36);
            float4 y = make_float4(0.f, 0.f, 0.f, 0.f);
            if (f0 + 32 * ((i >> 1) / NN) < rows) {
                y.x = k3d_act(gv.x, uv.x, b1, b2);
                y.y = k3d_act(gv.y, uv.y, b1, b2);
                y.z = k3d_act(gv.z, uv.z, b1, b2);
                y.w = k3d_act(gv.w, uv.w, b1, b2);
            }
            *(float4 *)o = y;
        }
        gm_wave_sync();
        const int col = 16 * (N0 + q4 % NN) + c16, b = q4 / NN;
        if (b < RG / 4 && col < np) {
            const float *o = wl + lane * 72;
            gm_v16f ev, od;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float4 v = *(const float4 *)(o + 4 * i);
                ev[2 * i] = v.x; od[2 * i] = v.y; ev[2 * i + 1] = v.z; od[2 * i + 1] = v.w;
            }
            const int f = f0 + 32 * b;
            if (gm_store_block(ev, od, h + ((size_t)(p0 + col) * nQh + (f >> 9)) * K3G_P6_QUAD, more,
                               gm_eight<false>(ev, od), (f >> 7) & 3, (f >> 5) & 3)) {
                wrow[p0 + col] = 1;
                *wide = 1;
            }
        }
        gm_wave_sync();
    };
    /* at most four (feature block, column block) pairs at a time */
    constexpr int PER = RG / 4 * NBW <= 4 ? NBW : 16 / RG;
    finish(GmInt<0>{}, GmInt<PER>{});
    if constexpr (NBW > PER) finish(GmInt<PER>{}, GmInt<(NBW - PER < PER ? NBW - PER : PER)>{});
    if constexpr (NBW > 2 * PER) {
        static_assert(NBW <= 3 * PER, "rounds");
        finish(GmInt<2 * PER>{}, GmInt<NBW - 2 * PER>{});
    }
}
