/*
 * k_gemm_bf16.hip — BF16-weight GEMM on MFMA (gfx950): Y [M, N] =
 * bf16(X [M, K] . W [N, K]^T), the bf16_gemm hook (c/bf16.h:712-767) for
 * more activation rows than a few passes of the streaming GEMV.
 *
 * A workgroup of 4 waves owns 64 RB activation rows x 64 CB weight rows; wave
 * (wr, wc) = (w / 2, w % 2) computes its 32 RB x 32 CB quarter with
 * v_mfma_f32_32x32x16_bf16, the weights as the A operand and the activations
 * as the B operand, so a lane ends with four consecutive output columns of
 * one row. K is walked in stages of 64 (whole 128-byte lines of both
 * matrices) through a ring of NS stages filled by direct global -> LDS loads;
 * 16-byte piece p of row r lies at p ^ ((r >> 1) & 7), which the operand
 * reads hit without bank conflicts. Operands are read D MFMA steps (of 4 a
 * stage) ahead; the one barrier of a stage sits at step 4 - D, after the
 * last read of the stage, and frees its buffer for stage j + NS at once.
 * Rows past M or N re-read the last row: computed, never stored.
 *
 * What bounds it: by the measured stage times, LDS. Over all tile shapes a
 * stage takes the direct loads' LDS writes at 64 B/clk plus the operand reads
 * at 128 B/clk (64 x 64: 540 clk, 128 x 128: 1000, 256 x 128: 1580), more than
 * its MFMAs (128, 512, 1024). The counters agree on the matrix cores (busy 47%
 * of the cycles at M = 2048, 29% at 600) and count the operand reads alone
 * (19% and 21%, conflicts 2-3% of those). Larger tiles read fewer LDS bytes per product, smaller ones fill
 * the chip at fewer rows: bg_pick chooses by those stage times.
 * Measured (rotating three sets of operands): M = 600, 4096 x 4096: 29 us,
 * 691 TFLOP/s (901 us as 150 GEMV passes of 4 rows); M = 2048: 60 us, 1144
 * TFLOP/s (3063 us).
 */
#include "ghip_device.h"
#include "ghip_internal.h"

#include <type_traits>

typedef float bg_f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int bg_u32x2 __attribute__((ext_vector_type(2)));

#define BG_LDS_MAX (160u * 1024u)

template <int RB, int CB, int D, int NS>
__global__ __launch_bounds__(256, 1) void k_bf16_gemm(const uint16_t *__restrict__ W,
                                                      const uint16_t *__restrict__ X,
                                                      uint16_t *__restrict__ Y, uint32_t M,
                                                      uint32_t N, uint32_t K, uint32_t mt) {
    constexpr uint32_t BM = 64u * RB, BN = 64u * CB;
    constexpr uint32_t ASTG = BM * 128u, STG = (BM + BN) * 128u;
    constexpr uint32_t NAL = BM / 32u, NWL = BN / 32u, LPS = NAL + NWL;
    static_assert(D == 1 || D == 2, "prefetch distance");
    static_assert(NS >= 2 && LPS * (NS - 1) <= 63 && NS * STG <= BG_LDS_MAX, "ring");
    constexpr int NSET = 2 * D;
    extern __shared__ __attribute__((aligned(1024))) uint8_t bg_lds[];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wr = wv >> 1, wc = wv & 1u;
    const uint32_t n = lane & 31u, h = lane >> 5;

    /* tile t: rows fastest, then columns; the workgroups of one XCD (b % 8)
     * take a run of consecutive tiles, so a column block's weights are read
     * into one XCD's L2 */
    uint32_t t;
    {
        const uint32_t T = gridDim.x, x = blockIdx.x & 7u, i = blockIdx.x >> 3;
        const uint32_t q = T >> 3, r = T & 7u;
        t = x * q + (x < r ? x : r) + i;
    }
    const uint32_t ct = t / mt, row0 = (t - ct * mt) * BM, col0 = ct * BN;
    const uint32_t rows = min(M - row0, BM), cols = min(N - col0, BN);
    const uint32_t nst = K >> 6;
    const uint8_t *xb = (const uint8_t *)(X + (size_t)row0 * K);
    const uint8_t *wb = (const uint8_t *)(W + (size_t)col0 * K);

    /* direct-load sources: load i of wave wv fills rows 8q .. 8q + 7, q = wv +
     * 4i, lane l's 16 bytes going to row 8q + l / 8, slot l % 8 */
    uint32_t aofs[NAL], wofs[NWL];
#pragma unroll
    for (uint32_t i = 0; i < NAL; i++) {
        const uint32_t r = 8u * (wv + 4u * i) + (lane >> 3);
        aofs[i] = min(r, rows - 1u) * K * 2u + 16u * ((lane & 7u) ^ ((r >> 1) & 7u));
    }
#pragma unroll
    for (uint32_t i = 0; i < NWL; i++) {
        const uint32_t r = 8u * (wv + 4u * i) + (lane >> 3);
        wofs[i] = min(r, cols - 1u) * K * 2u + 16u * ((lane & 7u) ^ ((r >> 1) & 7u));
    }
    /* part P of 4 of stage j's loads (P = -1: all of them) */
    auto issue = [&](auto part_c, uint32_t j) {
        constexpr int P = decltype(part_c)::value;
        uint8_t *st = bg_lds + (j % NS) * STG;
        const uint8_t *xj = xb + (size_t)j * 128u, *wj = wb + (size_t)j * 128u;
#pragma unroll
        for (uint32_t i = 0; i < NAL; i++)
            if (P < 0 || (int)(i & 3u) == P) ghip_dma16(xj + aofs[i], st + (wv + 4u * i) * 1024u);
#pragma unroll
        for (uint32_t i = 0; i < NWL; i++)
            if (P < 0 || (int)((NAL + i) & 3u) == P)
                ghip_dma16(wj + wofs[i], st + ASTG + (wv + 4u * i) * 1024u);
    };
    /* step s of lane half h takes k = 32h + 8s + [0, 8) of the stage from both
     * operands */
    uint32_t off[4];
#pragma unroll
    for (uint32_t s = 0; s < 4; s++) off[s] = n * 128u + 16u * ((4u * h + s) ^ ((n >> 1) & 7u));
    const uint32_t abase = wr * (32u * RB * 128u), wbase = ASTG + wc * (32u * CB * 128u);

    bg_f32x16 acc[RB][CB];
#pragma unroll
    for (int r = 0; r < RB; r++)
#pragma unroll
        for (int c = 0; c < CB; c++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[r][c][i] = 0.0f;
    ghip_bf16x8 xa[NSET][RB], wa[NSET][CB];
    auto fetch = [&](int set, uint32_t j, int s) {
        const uint8_t *st = bg_lds + (j % NS) * STG;
#pragma unroll
        for (int r = 0; r < RB; r++)
            xa[set][r] = *(const ghip_bf16x8 *)(st + abase + r * 4096u + off[s]);
#pragma unroll
        for (int c = 0; c < CB; c++)
            wa[set][c] = *(const ghip_bf16x8 *)(st + wbase + c * 4096u + off[s]);
    };
    using PA = std::integral_constant<int, -1>;
    /* all NS stages in flight, then the first D steps of stage 0 */
#pragma unroll
    for (uint32_t i = 0; i < NS; i++)
        if (i < nst) issue(PA{}, i);
    ghip_wait_stages<LPS, NS - 1>(nst - 1u);
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int s = 0; s < D; s++) fetch(s, 0u, s);

    /* MAIN: stage j + NS exists and is loaded during stage j. Without it the
     * waits shrink with the stages left, and the last stage's reads ahead
     * re-read the stage itself (unused) */
    auto stage = [&](uint32_t j, auto main_c) {
        constexpr bool MAIN = decltype(main_c)::value;
        const uint32_t jn = MAIN ? j + 1u : min(j + 1u, nst - 1u);
#pragma unroll
        for (int s = 0; s < 4; s++) {
            if (s == 4 - D) {
                /* own loads of stage j + 1 done, own reads of stage j done;
                 * after the barrier that holds for every wave */
                if (MAIN) GHIP_VMCNT(LPS * (NS - 2));
                else ghip_wait_stages<LPS, NS - 2>(nst - 1u - jn);
                __builtin_amdgcn_s_waitcnt(0xc07f);
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
            }
            if (MAIN && D == 1 && s == 3) issue(PA{}, j + NS);
            if (MAIN && D == 2 && s == 2) {
                issue(std::integral_constant<int, 0>{}, j + NS);
                issue(std::integral_constant<int, 1>{}, j + NS);
            }
            if (MAIN && D == 2 && s == 3) {
                issue(std::integral_constant<int, 2>{}, j + NS);
                issue(std::integral_constant<int, 3>{}, j + NS);
            }
            const int cur = s % NSET, nxt = (s + D) % NSET;
            if (s + D < 4) fetch(nxt, j, s + D);
            else fetch(nxt, jn, s + D - 4);
#pragma unroll
            for (int r = 0; r < RB; r++)
#pragma unroll
                for (int c = 0; c < CB; c++)
                    acc[r][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wa[cur][c], xa[cur][r],
                                                                       acc[r][c], 0, 0, 0);
            if (RB * CB >= RB + CB) {
#pragma unroll
                for (int i = 0; i < RB * CB; i++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    if (i < RB + CB) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    uint32_t j = 0;
    for (; j + NS < nst; j++) stage(j, std::true_type{});
    for (; j < nst; j++) stage(j, std::false_type{});

    /* epilogue: register 4q + i of block (r, c) is row 32r + n, column 32c +
     * 8q + 4h + i of the wave's quarter. Staged through a wave-private LDS
     * area (over the ring, once every wave has read it) so that the stores
     * are 16-byte vectors along a row; 2-byte stores where N or y do not
     * allow vectors */
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_s_barrier();
    constexpr uint32_t RBY = 64u * CB;                 /* bytes per staged row */
    constexpr uint32_t PM = 4u * CB - 1u;
    uint8_t *sw = bg_lds + wv * (32u * RB * RBY);
    const bool vec = (N & 7u) == 0u && ((uintptr_t)Y & 15u) == 0u;
#pragma unroll
    for (int r = 0; r < RB; r++)
#pragma unroll
        for (int c = 0; c < CB; c++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
                typedef float f4 __attribute__((ext_vector_type(4)));
                f4 v;
#pragma unroll
                for (int i = 0; i < 4; i++) v[i] = acc[r][c][4 * q + i];
                const bg_u32x2 b = __builtin_bit_cast(bg_u32x2, __builtin_convertvector(v, bf4));
                const uint32_t row = 32u * r + n;
                *(bg_u32x2 *)(sw + row * RBY + 16u * ((4u * c + q) ^ (row & PM)) + 8u * h) = b;
            }
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < 2 * RB * CB; i++) {
        const uint32_t v = lane + 64u * i, row = v / (4u * CB), p = v % (4u * CB);
        const ghip_u32x4 d = *(const ghip_u32x4 *)(sw + row * RBY + 16u * (p ^ (row & PM)));
        const uint32_t m = wr * (32u * RB) + row, c = wc * (32u * CB) + 8u * p;
        if (m < rows) {
            uint16_t *yp = Y + (size_t)(row0 + m) * N + col0 + c;
            if (vec) {
                if (c < cols) *(ghip_u32x4 *)yp = d;
            } else {
#pragma unroll
                for (uint32_t e = 0; e < 8; e++)
                    if (c + e < cols) yp[e] = (uint16_t)(d[e >> 1] >> (16u * (e & 1u)));
            }
        }
    }
}

/* One launchable tile shape. cost: measured microseconds of one tile over 64
 * stages (K = 4096) on an otherwise empty chip. */
struct BgTile {
    uint32_t bm, bn;
    float cost;
    const void *kern;
    uint32_t lds;
    void (*launch)(uint32_t, uint32_t, hipStream_t, hipEvent_t, hipEvent_t, const uint16_t *,
                   const uint16_t *, uint16_t *, uint32_t, uint32_t, uint32_t, uint32_t);
};

template <int RB, int CB, int D, int NS>
static void bg_run(uint32_t grid, uint32_t lds, hipStream_t st, hipEvent_t e0, hipEvent_t e1,
                   const uint16_t *w, const uint16_t *x, uint16_t *y, uint32_t M, uint32_t N,
                   uint32_t K, uint32_t mt) {
    GHIP_LAUNCH(e0, e1, (k_bf16_gemm<RB, CB, D, NS>), dim3(grid), dim3(256), lds, st, w, x, y, M,
                N, K, mt);
}

#define BG_TILE(RB, CB, D, NS, COST)                                                     \
    {64u * RB, 64u * CB, COST, (const void *)k_bf16_gemm<RB, CB, D, NS>,                 \
     NS * (64u * RB + 64u * CB) * 128u, bg_run<RB, CB, D, NS>}

static const BgTile bg_tiles[] = {
    BG_TILE(1, 1, 2, 8, 15.4f), BG_TILE(1, 2, 2, 6, 20.1f),
    BG_TILE(3, 1, 2, 5, 25.0f), BG_TILE(2, 2, 2, 5, 27.5f), BG_TILE(3, 2, 2, 4, 34.0f),
    BG_TILE(4, 2, 2, 3, 45.5f), BG_TILE(4, 4, 1, 2, 85.0f),
};

/* The tile shape with the least estimated time: rounds of the chip times the
 * tile's cost, up to 30% more as the round fills (every CU then shares the
 * caches and the clock; measured 29.1 against 27.5 us with 160 of 256 CUs
 * busy, 35.1 with all). The estimate is within 10% of the measured time over
 * M = 32..2048, N = 288..8192 for every shape. */
static const BgTile *bg_pick(size_t M, size_t N, uint32_t n_cu, double *est) {
    const BgTile *best = nullptr;
    double bc = 0.0;
    for (const BgTile &t : bg_tiles) {
        const double items = (double)((M + t.bm - 1) / t.bm) * (double)((N + t.bn - 1) / t.bn);
        const double rounds = (double)(size_t)((items + n_cu - 1) / n_cu);
        const double c = rounds * t.cost * (1.0 + 0.3 * items / (rounds * n_cu));
        if (!best || c < bc) {
            best = &t;
            bc = c;
        }
    }
    *est = bc;
    return best;
}

/* 32-bit offsets inside a tile (at most 256 rows of 2 K bytes) and a grid
 * below 2^31 workgroups. */
extern "C" int ghip_bf16_gemm_fits(size_t M, size_t N, size_t K, const void *w, const void *x) {
    return M > 0 && N > 0 && K > 0 && K % 64 == 0 && K <= ((size_t)1 << 22)
        && M <= 0x7fffffffu && N <= 0x7fffffffu
        && ((M + 63) / 64) * ((N + 63) / 64) <= 0x7fffffffu
        && ((uintptr_t)w & 15) == 0 && ((uintptr_t)x & 15) == 0;
}

/* Estimated microseconds: 3 + the pick's stages scaled to K (600 x 4096: 29.1
 * us at K = 4096, 17.1 at 2048), and no less than the weights at 5.7 TB/s
 * (LM head, M = 12: 225 us). */
extern "C" float ghip_bf16_gemm_estimate(size_t M, size_t N, size_t K, uint32_t n_cu) {
    double est = 0.0;
    (void)bg_pick(M, N, n_cu, &est);
    const double t = (est - 2.0) * (double)K / 4096.0, hbm = 2.0 * (double)N * (double)K / 5.7e6;
    return (float)(3.0 + (t > hbm ? t : hbm));
}

extern "C" uint32_t ghip_bf16_gemm_form(size_t M, size_t N, uint32_t n_cu) {
    double est = 0.0;
    const BgTile *t = bg_pick(M, N, n_cu, &est);
    return t->bm << 16 | t->bn;
}

extern "C" hipError_t ghip_launch_bf16_gemm(const uint16_t *w, const uint16_t *x, uint16_t *y,
                                            size_t M, size_t N, size_t K, uint32_t n_cu,
                                            hipEvent_t e0, hipEvent_t e1, hipStream_t st) {
    if (!ghip_bf16_gemm_fits(M, N, K, w, x) || n_cu == 0) return hipErrorInvalidValue;
    double est = 0.0;
    const BgTile *t = bg_pick(M, N, n_cu, &est);
    const size_t mt = (M + t->bm - 1) / t->bm, nt = (N + t->bn - 1) / t->bn;
    t->launch((uint32_t)(mt * nt), t->lds, st, e0, e1, w, x, y, (uint32_t)M, (uint32_t)N,
              (uint32_t)K, (uint32_t)mt);
    return hipGetLastError();
}

extern "C" hipError_t ghip_bf16_gemm_init(void) {
    for (const BgTile &t : bg_tiles) {
        hipError_t e = hipFuncSetAttribute(t.kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)t.lds);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
