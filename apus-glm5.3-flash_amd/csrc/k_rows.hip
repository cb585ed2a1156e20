/*
 * k_rows.hip — weight-streaming linear for a few activation rows (gfx950):
 * Y [M, N] = bf16(X [M, K] . W [N, K]^T) with FP8-block weights (c/gdsa.h:
 * 525-534) or BF16 ones (c/bf16.h:712-767), from one decode row over
 * speculative verifies and short prompts to a few dozen rows.
 *
 * A wave owns NT groups of 16 weight rows and, with KS waves splitting K, a
 * run of 128-byte-wide chunks of them. Per chunk it loads the weights (two
 * whole-line 16-byte loads a lane per group) and the same k range of MR rows
 * of x (1 KB loads: 4 rows of 256 bytes against FP8 codes, 8 of 128 against
 * BF16) into registers, writes both to a wave-private LDS slot and reads
 * them back in the layout of v_mfma_f32_16x16x32_bf16; NA chunks are in
 * flight. No barrier until the KS partial sums meet in LDS, added in a fixed
 * order (deterministic). Streaming x beside the weights, instead of staging
 * all of it first, takes any M x K; the weights are read once per MR rows.
 * LDS pieces are XOR-swizzled by row so the operand reads hit distinct banks.
 * Rows past M or N re-read the last row: computed, never stored.
 *
 * What bounds it: HBM for the larger weights (LM head 154880 x 4096, M = 1:
 * 180 us, 7.1 TB/s; o_proj 4096 x 16384, M = 4: 11.9 us, 5.7 TB/s), else the
 * chunk round trip of a wave (rw_cfgs' chunk times; the LDS traffic of x
 * from 16 rows on) and ~2.3 us of launch, first load and reduction.
 * Against passes of <= 4 rows over the weights: o_proj M = 4 46.7 -> 11.9 us,
 * q_a 1536 x 4096 M = 11 13.3 -> 5.1, LM head M = 1 205 -> 180, M = 8
 * 411 -> 181; and against the MFMA GEMM, q_a M = 64 14.6 -> 7.5.
 */
#include "ghip_device.h"
#include "ghip_internal.h"

#include <type_traits>

#define RW_NW 8                  /* waves per workgroup */
#define RW_LDS_MAX (160u * 1024u)
/* a launch's row tiles (grid y) and workgroups along the weight rows (grid x:
 * under 2^32 threads); more take several launches */
#define RW_MAX_TILES ((size_t)65535)
#define RW_MAX_BLOCKS (GHIP_MAX_THREADS / (RW_NW * 64))

/* LDS: each wave's SL slots of x and weights; the partial sums reuse it */
template <bool BF, int MR, int NT, int SL>
__host__ __device__ constexpr uint32_t rw_wave_lds() {
    return SL * ((MR * (BF ? 128u : 256u) < 1024u ? 1024u : MR * (BF ? 128u : 256u)) + 2048u * NT);
}
template <bool BF, int MR, int NT, int SL>
constexpr uint32_t rw_lds() {
    const uint32_t ring = RW_NW * rw_wave_lds<BF, MR, NT, SL>();
    const uint32_t red = RW_NW * MR * 16u * NT * 4u;
    return ring > red ? ring : red;
}

template <bool BF, int MR, int NT, int KS, int NA, int SL>
__global__ __launch_bounds__(RW_NW * 64, 1) void k_rows_gemm(
    const uint8_t *__restrict__ W, const float *__restrict__ S, const uint16_t *__restrict__ X,
    uint16_t *__restrict__ Y, uint32_t M, uint32_t O, uint32_t K,
    const uint32_t *__restrict__ exact_flag, uint32_t blk0, uint32_t tile0) {
    constexpr uint32_t GPP = RW_NW / KS;                 /* row groups per workgroup */
    constexpr uint32_t MT = MR < 16 ? 1 : MR / 16;
    constexpr uint32_t XI = BF ? (MR < 8 ? 1 : MR / 8) : MR / 4;  /* x loads per chunk */
    constexpr uint32_t XROW = BF ? 128u : 256u;          /* x bytes of a row in a chunk */
    constexpr uint32_t XB = XI * 1024u, SLOT = XB + 2048u * NT;
    static_assert(SL * SLOT == rw_wave_lds<BF, MR, NT, SL>() &&
                      rw_lds<BF, MR, NT, SL>() <= RW_LDS_MAX, "LDS layout");
    static_assert(SL == 1 || SL == NA, "one LDS slot, or one per register set");
    extern __shared__ __attribute__((aligned(1024))) uint8_t rl[];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t n = lane & 15u, g = lane >> 4;
    uint8_t *ring = rl + wv * (SL * SLOT);
    const uint32_t KB = BF ? 2u * K : K;                 /* weight row stride, bytes */
    const uint32_t nch = KB >> 7, nkb = K >> 7;
    const uint32_t part = wv % KS, slot = wv / KS;
    const uint32_t c0 = part * nch / KS, c1 = (part + 1u) * nch / KS, nc = c1 - c0;
    const uint32_t blk = blk0 + blockIdx.x, grp = blk * GPP + slot, row0 = grp * (16u * NT);
    const uint32_t m0 = (tile0 + blockIdx.y) * MR;
    const uint32_t mrows = min(M - m0, (uint32_t)MR);
    ghip_f32x4 acc[MT][NT];
#pragma unroll
    for (uint32_t a = 0; a < MT; a++)
#pragma unroll
        for (int b = 0; b < NT; b++) acc[a][b] = (ghip_f32x4){0.f, 0.f, 0.f, 0.f};

    if (row0 < O && nc > 0u) {
        const uint8_t *rows = W + (size_t)row0 * KB;
        ghip_cdma d[NT];
#pragma unroll
        for (int b = 0; b < NT; b++) {
            const uint32_t left = O - 1u - row0;
            if (left >= 16u * b + 15u) {
                d[b] = ghip_cdma_offsets(lane, KB);
                d[b].off0 += 16u * b * KB;
                d[b].off1 += 16u * b * KB;
            } else {
                const uint32_t r0 = min(16u * b + (lane >> 3), left);
                const uint32_t r1 = min(16u * b + 8u + (lane >> 3), left);
                /* the piece swizzle is by the LDS row, not the clamped one */
                d[b].off0 = r0 * KB + 16u * ((lane & 7u) ^ ((lane >> 4) & 7u));
                d[b].off1 = r1 * KB + 16u * ((lane & 7u) ^ ((4u + (lane >> 4)) & 7u));
            }
        }
        /* x load u: BF rows 8u + l/8, piece l % 8; FP8 rows 4u + l/16, piece
         * l % 16 */
        constexpr uint32_t LPR = XROW / 16u;             /* lanes per row */
        const uint8_t *xb = (const uint8_t *)(X + (size_t)m0 * K);
        uint32_t xo[XI];
#pragma unroll
        for (uint32_t u = 0; u < XI; u++) {
            const uint32_t r = u * (64u / LPR) + lane / LPR;
            const uint32_t sw = BF ? (r >> 1) & 7u : r & 15u;
            xo[u] = min(r, mrows - 1u) * K * 2u + 16u * ((lane & (LPR - 1u)) ^ sw);
        }
        ghip_u32x4 xr[NA][XI], wr[NA][2 * NT];
        auto load = [&](auto set_c, uint32_t c) {
            constexpr int A = decltype(set_c)::value;
            const uint8_t *xc = xb + (size_t)c * XROW, *wc = rows + (size_t)c * 128u;
#pragma unroll
            for (uint32_t u = 0; u < XI; u++) xr[A][u] = *(const ghip_u32x4 *)(xc + xo[u]);
#pragma unroll
            for (int b = 0; b < NT; b++) {
                wr[A][2 * b] = __builtin_nontemporal_load((const ghip_u32x4 *)(wc + d[b].off0));
                wr[A][2 * b + 1] = __builtin_nontemporal_load((const ghip_u32x4 *)(wc + d[b].off1));
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        const float *srow = BF ? nullptr : S + (size_t)(row0 >> 7) * nkb;
        const bool exact = !BF && exact_flag != nullptr && *exact_flag != 0u;
        auto step = [&](auto set_c, auto refill_c, uint32_t t) {
            constexpr int A = decltype(set_c)::value;
            uint8_t *xs = ring + (SL == 1 ? 0u : A * SLOT), *ws = xs + XB;
#pragma unroll
            for (uint32_t u = 0; u < XI; u++)
                *(ghip_u32x4 *)(xs + u * 1024u + lane * 16u) = xr[A][u];
#pragma unroll
            for (int b = 0; b < NT; b++)
                ghip_rl_store(ws + 2048u * b, lane, wr[A][2 * b], wr[A][2 * b + 1]);
            if constexpr (decltype(refill_c)::value) {
                __builtin_amdgcn_sched_barrier(0);
                load(set_c, c0 + t + NA);
            }
            ghip_chunk cw[NT];
#pragma unroll
            for (int b = 0; b < NT; b++) cw[b] = ghip_cdma_read(ws + 2048u * b, n, g);
            if constexpr (BF) {
#pragma unroll
                for (uint32_t a = 0; a < MT; a++) {
                    const uint32_t r = MR < 16 ? n & (MR - 1u) : 16u * a + n;
                    const uint32_t sw = (r >> 1) & 7u;
                    const ghip_bf16x8 x0 = *(const ghip_bf16x8 *)(xs + r * 128u + 16u * ((2u * g) ^ sw));
                    const ghip_bf16x8 x1 = *(const ghip_bf16x8 *)(xs + r * 128u + 16u * ((2u * g + 1u) ^ sw));
#pragma unroll
                    for (int b = 0; b < NT; b++) {
                        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            x0, __builtin_bit_cast(ghip_bf16x8, cw[b].lo), acc[a][b], 0, 0, 0);
                        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            x1, __builtin_bit_cast(ghip_bf16x8, cw[b].hi), acc[a][b], 0, 0, 0);
                    }
                }
            } else {
                const float sc = ghip_sload(srow, c0 + t);
                ghip_bf16x8 w4[NT][4];
#pragma unroll
                for (int b = 0; b < NT; b++) {
                    if (exact) {
                        ghip_deq16<true>(cw[b].lo, sc, w4[b][0], w4[b][1]);
                        ghip_deq16<true>(cw[b].hi, sc, w4[b][2], w4[b][3]);
                    } else {
                        ghip_deq16<false>(cw[b].lo, sc, w4[b][0], w4[b][1]);
                        ghip_deq16<false>(cw[b].hi, sc, w4[b][2], w4[b][3]);
                    }
                }
#pragma unroll
                for (uint32_t a = 0; a < MT; a++) {
                    const uint32_t r = MR < 16 ? n & (MR - 1u) : 16u * a + n;
#pragma unroll
                    for (uint32_t i = 0; i < 4; i++) {
                        const ghip_bf16x8 xv = *(const ghip_bf16x8 *)(
                            xs + r * 256u + 16u * ((4u * g + i) ^ (r & 15u)));
#pragma unroll
                        for (int b = 0; b < NT; b++)
                            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xv, w4[b][i],
                                                                               acc[a][b], 0, 0, 0);
                    }
                }
            }
        };
        using RF = std::true_type;
        using NR = std::false_type;
        using S0 = std::integral_constant<int, 0>;
        using S1 = std::integral_constant<int, NA - 1>;
        load(S0{}, c0);
        if constexpr (NA == 2) load(S1{}, min(c0 + 1u, nch - 1u));
        uint32_t t = 0;
        if constexpr (NA == 1) {
            for (; t + 1u < nc; t++) step(S0{}, RF{}, t);
            step(S0{}, NR{}, t);
        } else {
            for (; t + 3u < nc; t += 2u) {
                step(S0{}, RF{}, t);
                step(S1{}, RF{}, t + 1u);
            }
            if (nc - t == 3u) {
                step(S0{}, RF{}, t);
                step(S1{}, NR{}, t + 1u);
                step(S0{}, NR{}, t + 2u);
            } else if (nc - t == 2u) {
                step(S0{}, NR{}, t);
                step(S1{}, NR{}, t + 1u);
            } else {
                step(S0{}, NR{}, t);
            }
        }
    }
    /* the KS partial sums of each group, added in order */
    __syncthreads();
    float *red = (float *)rl;                            /* [8 waves][MR][16 NT] */
#pragma unroll
    for (uint32_t a = 0; a < MT; a++)
#pragma unroll
        for (int b = 0; b < NT; b++)
#pragma unroll
            for (uint32_t i = 0; i < 4; i++) {
                const uint32_t m = 16u * a + 4u * g + i;
                if (MR >= 16 || m < (uint32_t)MR)
                    red[(wv * MR + m) * (16u * NT) + 16u * b + n] = acc[a][b][i];
            }
    __syncthreads();
    for (uint32_t v = tid; v < GPP * MR * 16u * NT; v += RW_NW * 64u) {
        const uint32_t sl = v / (MR * 16u * NT), e = v - sl * (MR * 16u * NT);
        const uint32_t m = e / (16u * NT), c = e - m * (16u * NT);
        const uint32_t o = (blk * GPP + sl) * (16u * NT) + c;
        if (m < mrows && o < O) {
            float s = 0.0f;
#pragma unroll
            for (int k = 0; k < KS; k++) s += red[((sl * KS + k) * MR) * (16u * NT) + e];
            Y[(size_t)(m0 + m) * O + o] = (uint16_t)ghip_bf16_bits(s);
        }
    }
}

/* One launchable form: MR rows of x, NT groups of 16 weight rows per wave, K
 * over KS waves. chunk: measured microseconds of a wave's chunk step. */
struct RwCfg {
    uint32_t mr, nt, ks;
    float chunk;
    const void *kern;
    uint32_t lds;
    void (*launch)(dim3, uint32_t, hipStream_t, hipEvent_t, hipEvent_t, const uint8_t *,
                   const float *, const uint16_t *, uint16_t *, uint32_t, uint32_t, uint32_t,
                   const uint32_t *, uint32_t, uint32_t);
};

template <bool BF, int MR, int NT, int KS, int NA, int SL>
static void rw_run(dim3 grid, uint32_t lds, hipStream_t st, hipEvent_t e0, hipEvent_t e1,
                   const uint8_t *w, const float *s, const uint16_t *x, uint16_t *y, uint32_t M,
                   uint32_t O, uint32_t K, const uint32_t *exact, uint32_t blk0,
                   uint32_t tile0) {
    GHIP_LAUNCH(e0, e1, (k_rows_gemm<BF, MR, NT, KS, NA, SL>), grid, dim3(RW_NW * 64), lds, st, w,
                s, x, y, M, O, K, exact, blk0, tile0);
}

#define RW_CFG(BF, MR, NT, KS, NA, SL, T)                                                  \
    {MR, NT, KS, T, (const void *)k_rows_gemm<BF, MR, NT, KS, NA, SL>, rw_lds<BF, MR, NT, SL>(), \
     rw_run<BF, MR, NT, KS, NA, SL>}

/* Two chunks in flight up to 16 rows of x (o_proj, M = 8: 14.0 us against
 * 14.9 with one), one where x's registers and LDS slots grow past that
 * (q_a, M = 32: 7.6 against 8.0 with two). */
static const RwCfg rw_fp8[] = {
    RW_CFG(false, 4, 1, 8, 2, 2, 0.55f),  RW_CFG(false, 4, 1, 4, 2, 2, 0.55f),
    RW_CFG(false, 4, 1, 2, 2, 2, 0.56f),  RW_CFG(false, 8, 1, 8, 2, 2, 0.65f),
    RW_CFG(false, 8, 1, 4, 2, 2, 0.65f),  RW_CFG(false, 8, 1, 2, 2, 2, 0.62f),
    RW_CFG(false, 16, 1, 8, 1, 1, 0.85f), RW_CFG(false, 16, 2, 8, 2, 2, 1.30f),
    RW_CFG(false, 16, 2, 4, 2, 2, 1.30f), RW_CFG(false, 32, 1, 8, 1, 1, 1.30f),
    RW_CFG(false, 32, 2, 8, 1, 1, 1.70f), RW_CFG(false, 32, 2, 4, 1, 1, 1.70f),
    RW_CFG(false, 64, 2, 4, 1, 1, 2.20f),
};
static const RwCfg rw_bf16[] = {
    RW_CFG(true, 8, 1, 8, 2, 2, 0.50f),  RW_CFG(true, 8, 1, 4, 2, 2, 0.50f),
    RW_CFG(true, 16, 1, 8, 2, 2, 0.58f), RW_CFG(true, 16, 1, 4, 2, 2, 0.60f),
    RW_CFG(true, 16, 2, 4, 2, 2, 0.75f), RW_CFG(true, 32, 1, 8, 1, 1, 0.85f),
    RW_CFG(true, 32, 2, 8, 1, 1, 1.20f), RW_CFG(true, 32, 2, 4, 1, 1, 1.15f),
};

/* Estimated microseconds of a form: 2.3 + the larger of rounds of the chip x
 * a wave's chunks x the chunk time and the weights at 6.5 TB/s + a tenth of
 * the other (within 20% of the measured times over M = 1..192 and the shapes
 * above). Where the weights' bytes decide, the form with less LDS a workgroup
 * is the better one by a few percent (more workgroups a CU; LM head, M = 1:
 * 8 rows x 1 group 178 us, 16 x 2 184). Forms of 4 and 8 rows only take as
 * many: more row tiles would re-read the weights. */
static float rw_estimate(const RwCfg &c, bool bf, size_t M, size_t N, size_t K, uint32_t n_cu) {
    if (c.mr < 16 && M > c.mr) return 1e30f;
    const double gpp = 16.0 * c.nt * (RW_NW / c.ks);
    const double wgs = (double)(size_t)((N + gpp - 1) / gpp) * (double)((M + c.mr - 1) / c.mr);
    const double nch = (double)(bf ? 2 * K : K) / 128.0;
    const double rounds = (double)(size_t)((wgs + n_cu - 1) / n_cu);
    const double nc = (double)(size_t)((nch + c.ks - 1) / c.ks);
    const double hbm = (double)N * (double)(bf ? 2 * K : K) / 6.5e6;
    /* A round's first loads and reduction: hidden under no other workgroup by
     * the form of 64 rows (16384 x 1536: 13.4 us at M = 64 in one round, 25.4
     * at 128 in two, where the MFMA GEMM takes 21.5), and past the first round
     * of other FP8 forms with two or more blocks where a wave has few chunks
     * (32768 x 1024: M = 48 in six rounds of 16 rows 37.9 us, M = 64 in four
     * of 32 27.5, the GEMM 16.6 and 18; 16384 x 1536, M = 80, three rounds 22,
     * the GEMM 20.5). */
    const double over = c.mr > 32 ? 3.8 * rounds
                        : !bf && c.mr * c.nt >= 32 && nc < 8.0 ? 2.0 * (rounds - 1.0)
                                                         : 0.0;
    const double t = rounds * nc * c.chunk + over;
    const double lds = t < hbm ? 0.0015 * hbm * c.mr * c.nt : 0.0;
    return (float)(2.3 + (t > hbm ? t + 0.1 * hbm : hbm + 0.1 * t) + lds);
}

static const RwCfg *rw_pick(bool bf, size_t M, size_t N, size_t K, uint32_t n_cu, float *est) {
    const RwCfg *best = nullptr;
    const RwCfg *tab = bf ? rw_bf16 : rw_fp8;
    const size_t n = bf ? sizeof rw_bf16 / sizeof *rw_bf16 : sizeof rw_fp8 / sizeof *rw_fp8;
    for (size_t i = 0; i < n; i++) {
        const float c = rw_estimate(tab[i], bf, M, N, K, n_cu);
        if (!best || c < *est) {
            best = &tab[i];
            *est = c;
        }
    }
    return best;
}

/* 32-bit offsets inside a wave's rows */
extern "C" int ghip_rows_fits(int bf, size_t M, size_t N, size_t K, const void *w, const void *x) {
    return M > 0 && M <= 0x7fffffffu && N > 0 && N <= 0x7fffffffu && K > 0
        && K <= ((size_t)1 << 24) && K % (bf ? 64 : 128) == 0 && ((uintptr_t)w & 15) == 0
        && ((uintptr_t)x & 15) == 0;
}

extern "C" float ghip_rows_estimate(int bf, size_t M, size_t N, size_t K, uint32_t n_cu) {
    float est = 0.0f;
    (void)rw_pick(bf != 0, M, N, K, n_cu, &est);
    return est;
}

extern "C" uint32_t ghip_rows_form(int bf, size_t M, size_t N, size_t K, uint32_t n_cu) {
    float est = 0.0f;
    const RwCfg *c = rw_pick(bf != 0, M, N, K, n_cu, &est);
    return c->mr << 16 | c->nt << 8 | c->ks;
}

extern "C" hipError_t ghip_launch_rows(int bf, const void *w, const float *scales,
                                       const uint16_t *x, uint16_t *y, size_t M, size_t N,
                                       size_t K, const uint32_t *exact_dev, uint32_t n_cu,
                                       hipEvent_t e0, hipEvent_t e1, hipStream_t st) {
    if (!ghip_rows_fits(bf, M, N, K, w, x) || n_cu == 0) return hipErrorInvalidValue;
    float est = 0.0f;
    const RwCfg *c = rw_pick(bf != 0, M, N, K, n_cu, &est);
    const size_t gpp = 16u * c->nt * (RW_NW / c->ks), blocks = (N + gpp - 1) / gpp;
    const size_t tiles = (M + c->mr - 1) / c->mr;
    for (size_t t0 = 0; t0 < tiles; t0 += RW_MAX_TILES)
        for (size_t b0 = 0; b0 < blocks; b0 += RW_MAX_BLOCKS) {
            const size_t nt = tiles - t0 < RW_MAX_TILES ? tiles - t0 : RW_MAX_TILES;
            const size_t nb = blocks - b0 < RW_MAX_BLOCKS ? blocks - b0 : RW_MAX_BLOCKS;
            c->launch(dim3((uint32_t)nb, (uint32_t)nt), c->lds, st,
                      t0 == 0 && b0 == 0 ? e0 : nullptr,
                      t0 + nt == tiles && b0 + nb == blocks ? e1 : nullptr, (const uint8_t *)w,
                      scales, x, y, (uint32_t)M, (uint32_t)N, (uint32_t)K, exact_dev,
                      (uint32_t)b0, (uint32_t)t0);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) return e;
        }
    return hipSuccess;
}

extern "C" hipError_t ghip_rows_init(void) {
    for (const RwCfg &c : rw_fp8) {
        hipError_t e = hipFuncSetAttribute(c.kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)c.lds);
        if (e != hipSuccess) return e;
    }
    for (const RwCfg &c : rw_bf16) {
        hipError_t e = hipFuncSetAttribute(c.kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)c.lds);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
