/*
 * k_linear.hip — gfx950 kernels for the dense FP8-block path:
 *   K2  k_fp8_gemv_stream : decode / MTP-verify GEMV (M <= 4) of many FP8
 *       weight rows, with the dequant fused in registers and the k reduction
 *       on MFMA (v_mfma_f32_16x16x32_bf16), the composition of
 *       c/gdsa.h:525-534 (dequant -> bf16 -> fp32-accumulated GEMM -> RNE
 *       bf16), and of few long BF16 ones (c/bf16.h:712-767). Other row counts
 *       and shapes: k_rows.hip, k_moe_prefill.hip (k_fp8_gemm) and, for BF16
 *       weights, k_gemm_bf16.hip.
 *   k_linear_any : shape-general fallback (K not a multiple of 128 / 64,
 *       unaligned operands) with the exact integer decode.
 *   k_nan_scan : flags the out-of-contract NaN codes 0x7F/0xFF so callers
 *       can select the exact decode for such weights.
 *
 * The MFMA k-slot to k mapping is any permutation used identically for A and
 * B, so a result is an exact-product fp32 sum in a different order than the
 * reference's sequential k: a tolerance-class result, per the contract.
 * Partial sums of waves are combined in LDS in a fixed order, so outputs are
 * deterministic run to run.
 */
#include "ghip_device.h"
#include <type_traits>
#include "ghip_internal.h"

/* NaN-code scan: bytes whose low 7 bits are all ones (0x7F / 0xFF). */
__global__ __launch_bounds__(256) void k_nan_scan(
    const uint8_t *__restrict__ p, size_t n, uint32_t *flag) {
    const size_t nv = n >> 4;
    uint32_t hit = 0;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < nv;
         i += (size_t)gridDim.x * 256) {
        ghip_u32x4 v = *(const ghip_u32x4 *)(p + (i << 4));
        for (int j = 0; j < 4; j++)
            hit |= ((v[j] & 0x7f7f7f7fu) + 0x01010101u) & 0x80808080u;
    }
    if (blockIdx.x == 0)
        for (size_t i = (nv << 4) + threadIdx.x; i < n; i += 256)
            hit |= ((p[i] & 0x7fu) == 0x7fu);
    if (hit) atomicOr(flag, 1u);
}

/* ------------------------------------------------------------------------ */
/* shape-general fallback: exact decode                                     */
/* ------------------------------------------------------------------------ */

__device__ __forceinline__ float wave_sum(float v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

/* One wave per weight row and MR rows of x: the decode and the weight's loads
 * serve all of them, and the loads of four k steps are in flight together. Each
 * sum is its lanes' k = lane, lane + 64, ... in order and then the wave's, for
 * any MR. Bound by issue (any alignment: loads of one element): 2000 x 2001, M
 * = 64, weights from HBM, FP8 52 us and BF16 37 (a wave a row of x 222 and
 * 147), M = 3 15.0 and 5.9 (22.7 and 12.5, each load waited for). */
template <bool BF, int MR>
__global__ __launch_bounds__(256) void k_linear_any(
    const void *__restrict__ W, const float *__restrict__ S,
    const uint16_t *__restrict__ X, uint16_t *__restrict__ Y, uint32_t M,
    uint32_t O, uint32_t K, uint32_t nkb, uint32_t blk0) {
    const uint32_t lane = threadIdx.x & 63u;
    const size_t item = ((size_t)blk0 + blockIdx.x) * 4 + (threadIdx.x >> 6);
    const uint32_t mt = (M + MR - 1u) / MR;
    if (item >= (size_t)mt * O) return;
    const uint32_t m0 = (uint32_t)(item / O) * MR, o = (uint32_t)(item % O);
    const uint8_t *wr = (const uint8_t *)W + (size_t)o * K * (BF ? 2u : 1u);
    const float *srow = BF ? nullptr : S + (size_t)(o >> 7) * nkb;
    const uint16_t *xr[MR];
#pragma unroll
    for (int i = 0; i < MR; i++) xr[i] = X + (size_t)min(m0 + i, M - 1u) * K;
    auto weight = [&](uint32_t k) -> float {
        if (BF) return ghip_bf16_f32(((const uint16_t *)wr)[k]);
        return ghip_bf16_round(ghip_e4m3_exact(wr[k]) * srow[k >> 7]);
    };
    float acc[MR] = {};
    /* U steps of 64 from k0; END: the last of them ends at K, and a lane past
     * it adds +0 */
    auto steps = [&](auto u_c, auto end_c, uint32_t k0) {
        constexpr int U = decltype(u_c)::value;
        constexpr bool END = decltype(end_c)::value;
        float wv[U], xv[U][MR];
#pragma unroll
        for (int j = 0; j < U; j++) {
            const bool last = END && j == U - 1;
            const uint32_t k = k0 + 64u * j + lane, kc = last ? min(k, K - 1u) : k;
            wv[j] = weight(kc);
            if (last) wv[j] = k < K ? wv[j] : 0.0f;
#pragma unroll
            for (int i = 0; i < MR; i++) {
                const float v = ghip_bf16_f32(xr[i][kc]);
                xv[j][i] = last && k >= K ? 0.0f : v;
            }
        }
#pragma unroll
        for (int j = 0; j < U; j++)
#pragma unroll
            for (int i = 0; i < MR; i++) acc[i] += wv[j] * xv[j][i];
    };
    using ST = std::true_type;
    using SF = std::false_type;
    uint32_t k0 = 0;
    for (; K - k0 > 256u; k0 += 256u) steps(std::integral_constant<int, 4>{}, SF{}, k0);
    /* no more steps than K has: four for 1 of 257 cost up to a fifth (2000 x
     * 257, M = 3, FP8: 5.5 us against 4.7) */
    switch ((K - k0 + 63u) >> 6) {
    case 4: steps(std::integral_constant<int, 4>{}, ST{}, k0); break;
    case 3: steps(std::integral_constant<int, 3>{}, ST{}, k0); break;
    case 2: steps(std::integral_constant<int, 2>{}, ST{}, k0); break;
    default: steps(std::integral_constant<int, 1>{}, ST{}, k0); break;
    }
#pragma unroll
    for (int i = 0; i < MR; i++) {
        const float s = wave_sum(acc[i]);
        if (lane == 0 && m0 + i < M) Y[(size_t)(m0 + i) * O + o] = (uint16_t)ghip_bf16_bits(s);
    }
}

/* The most rows of x a wave (8, 4, 2) that leave 4096 waves, four a SIMD. */
template <bool BF>
static hipError_t launch_linear_any(const void *w, const float *s, const uint16_t *x, uint16_t *y,
                                    size_t M, size_t O, size_t K, hipEvent_t ev0, hipEvent_t ev1,
                                    hipStream_t st) {
    if (M * O > 0xffffffffull * 4) return hipErrorInvalidValue;
    const uint32_t nkb = (uint32_t)((K + 127) / 128);
    size_t mr = 8;
    while (mr > 1 && (mr > M || O * ((M + mr - 1) / mr) < 4096)) mr >>= 1;
    const size_t blocks = (O * ((M + mr - 1) / mr) + 3) / 4, most = GHIP_MAX_THREADS / 256u;
#define LINEAR_ANY(R) \
    GHIP_LAUNCH(b == 0 ? ev0 : nullptr, b + n == blocks ? ev1 : nullptr, (k_linear_any<BF, R>), \
                dim3((uint32_t)n), dim3(256), 0, st, w, s, x, y, (uint32_t)M, (uint32_t)O, \
                (uint32_t)K, nkb, (uint32_t)b)
    for (size_t b = 0; b < blocks; b += most) {
        const size_t n = blocks - b < most ? blocks - b : most;
        if (mr == 8) LINEAR_ANY(8);
        else if (mr == 4) LINEAR_ANY(4);
        else if (mr == 2) LINEAR_ANY(2);
        else LINEAR_ANY(1);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
#undef LINEAR_ANY
    return hipSuccess;
}

/* ------------------------------------------------------------------------ */
/* launchers                                                                */
/* ------------------------------------------------------------------------ */

static uint32_t grid_for(size_t items, size_t per_block, uint32_t cap) {
    size_t g = (items + per_block - 1) / per_block;
    if (g < 1) g = 1;
    if (g > cap) g = cap;
    return (uint32_t)g;
}

extern "C" hipError_t ghip_launch_nan_scan(const uint8_t *codes, size_t n,
                                           uint32_t *flag, hipStream_t st) {
    if (n == 0) return hipSuccess;
    if (((uintptr_t)codes & 15) != 0) return hipErrorInvalidValue;
    uint32_t g = grid_for(n / 16 + 1, 256 * 8, 4096);
    hipLaunchKernelGGL(k_nan_scan, dim3(g), dim3(256), 0, st, codes, n, flag);
    return hipGetLastError();
}

/* ------------------------------------------------------------------------ */
/* K2: persistent GEMV, M <= 4, x staged once, weights streamed             */
/* ------------------------------------------------------------------------ */

#define GS_NW 8                  /* waves per workgroup */
/* chunks in flight and LDS slots of a wave: a chunk is written from registers
 * and read back in the MFMA layout while the next ones are in flight (FP8,
 * 16384 x 4096: one 13.8 us, two 12.3, three 12.6) */
#define GS_NA(BF) ((BF) ? 3u : 2u)
#define GS_X_MAX (48u * 1024u)   /* FP8: most bytes of x staged (K <= 6144 at M = 4) */
#define GS_LDS (144u * 1024u)    /* dynamic LDS limit of the streaming GEMV */

/* Y[m, rows] for M <= 4 token rows. A row group (16 weight rows) is split
 * over KS waves along K (FP8 2, BF16 8); a workgroup pass covers 8 / KS row
 * groups, passes run over the groups persistently (at most one workgroup per
 * CU). Each wave streams its chunks (16 rows x 128 bytes: 128 codes, one scale
 * block, or 64 BF16 weights) through registers: two 16-byte loads per lane in
 * a whole-line pattern (load i: rows 8i + lane / 8, piece lane % 8), NA chunks
 * in flight, each chunk written to a wave-private LDS slot (lane l's bytes at
 * 16 l, piece p of row r at p ^ ((r >> 1) & 7)) and read back in the MFMA
 * layout, dequantized in registers (FP8) and reduced on MFMA with the token
 * rows of x (staged once per workgroup) as the A operand: A row i = lane % 16
 * is token min(i, M-1), rows past M feed output rows that are discarded. The
 * KS partial sums of a group are added in LDS in a fixed order
 * (deterministic). */
template <int M, int KS, bool BF>
__global__ __launch_bounds__(GS_NW * 64, 1) void k_fp8_gemv_stream(
    const uint8_t *__restrict__ W, const float *__restrict__ S,
    const uint16_t *__restrict__ X, uint16_t *__restrict__ Y, uint32_t O,
    uint32_t K, const uint32_t *__restrict__ exact_flag) {
    constexpr uint32_t GPP = GS_NW / KS;             /* row groups per pass */
    constexpr uint32_t NA = GS_NA(BF);               /* chunks in flight, LDS slots */
    extern __shared__ __attribute__((aligned(1024))) uint8_t gsl[];
    __shared__ float red[GPP][KS][M][16];
    uint16_t *xs = (uint16_t *)gsl;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t n = lane & 15u, g = lane >> 4;
    uint8_t *ring = gsl + (((size_t)M * K * 2u + 1023u) & ~(size_t)1023u) +
                    wv * (NA * 2048u);
    /* chunk = 128 bytes of each of 16 rows; row stride in bytes */
    const uint32_t KB = BF ? 2u * K : K;
    const uint32_t nch = KB >> 7, nkb = K >> 7;
    const uint32_t part = wv % KS, slot = wv / KS;
    const uint32_t c0 = part * nch / KS, c1 = (part + 1) * nch / KS, nc = c1 - c0;
    const uint32_t groups = (O + 15) / 16, passes = (groups + GPP - 1) / GPP;
    const uint16_t *xa = xs + (size_t)min(n, (uint32_t)M - 1u) * K + (BF ? 16u : 32u) * g;
    /* pass ps's row group of this wave: its rows and load offsets (a
     * partial last group re-reads row O-1, outputs discarded) */
    auto rows_of = [&](uint32_t ps) {
        return W + (size_t)(ps * GPP + slot) * 16u * KB;
    };
    auto offs_of = [&](uint32_t ps) {
        return ghip_cdma_offsets(lane, KB, min(15u, O - 1u - (ps * GPP + slot) * 16u));
    };
    /* chunk t's two 16-byte pieces in register set t % NA ((ra0, ra1), (rb0,
     * rb1), (rc0, rc1)) and LDS slot t % NA */
    ghip_u32x4 ra0, ra1, rb0, rb1, rc0, rc1;
    /* the first NA chunks of a pass, always all loaded (chunk indices
     * clamped): a fixed count of loads in flight, in a fixed order */
    auto prefetch = [&](const uint8_t *rows, const ghip_cdma &d) {
        ghip_rl_load(rows, d, min(c0, nch - 1u), ra0, ra1);
        __builtin_amdgcn_sched_barrier(0);
        ghip_rl_load(rows, d, min(c0 + 1u, nch - 1u), rb0, rb1);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (NA == 3u) {
            ghip_rl_load(rows, d, min(c0 + 2u, nch - 1u), rc0, rc1);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    /* x into LDS without delaying the weight stream: x goes by direct DMA
     * (1 K pieces dealt to the waves, lanes past x re-read its last vector
     * into the 1 K-rounded x region) ahead of the first pass's 2 NA chunk
     * loads, so waiting until no more than those are in flight means this
     * wave's x pieces have landed */
    {
        const uint32_t nvec = (uint32_t)M * (K >> 3), nxc = (nvec + 63u) >> 6;
        for (uint32_t c = wv; c < nxc; c += GS_NW)
            ghip_dma16(X + (size_t)min(c * 64u + lane, nvec - 1u) * 8u, gsl + c * 1024u);
        const uint32_t grp0 = min(blockIdx.x * GPP + slot, groups - 1u);
        prefetch(W + (size_t)grp0 * 16u * KB,
               ghip_cdma_offsets(lane, KB, min(15u, O - 1u - grp0 * 16u)));
        GHIP_VMCNT(2 * NA);
    }
    /* a bare barrier: __syncthreads() would also wait for the chunk loads
     * (its workgroup-scope release waits for every load in flight) */
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const bool exact = !BF && exact_flag != nullptr && *exact_flag != 0u;
    for (uint32_t ps = blockIdx.x; ps < passes; ps += gridDim.x) {
        const uint32_t grp = ps * GPP + slot;
        const bool live = grp < groups;
        if (live) {
            /* a wave with no chunks contributes zeros */
            const uint32_t row0 = grp * 16;
            const uint8_t *rows = rows_of(ps);
            const ghip_cdma d = offs_of(ps);
            const float *srow = BF ? nullptr : S + (size_t)(row0 >> 7) * nkb;
            if (ps != blockIdx.x) prefetch(rows, d);
            ghip_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
            /* chunk t: its registers into LDS slot t % NA, the registers
             * refilled with chunk t + NA (REFILL), the chunk read back in
             * the MFMA layout with this lane's activations and the scale */
            auto step = [&](auto refill_c, uint32_t t, ghip_u32x4 &v0, ghip_u32x4 &v1,
                            uint8_t *buf) {
                ghip_rl_store(buf, lane, v0, v1);
                if constexpr (decltype(refill_c)::value) {
                    __builtin_amdgcn_sched_barrier(0);
                    ghip_rl_load(rows, d, c0 + t + NA, v0, v1);
                    __builtin_amdgcn_sched_barrier(0);
                }
                const uint32_t c = c0 + t;
                const ghip_chunk cw = ghip_cdma_read(buf, n, g);
                if constexpr (BF) {
                    const ghip_bf16x8 *a = (const ghip_bf16x8 *)(xa + c * 64u);
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        a[0], __builtin_bit_cast(ghip_bf16x8, cw.lo), acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        a[1], __builtin_bit_cast(ghip_bf16x8, cw.hi), acc, 0, 0, 0);
                } else {
                    ghip_bf16x8 a4[4];
                    ghip_read_a4(xa + c * 128u, a4);
                    const float sc = ghip_sload(srow, c);
                    if (exact) ghip_chunk_mfma_a<true>(cw, sc, a4, acc);
                    else ghip_chunk_mfma_a<false>(cw, sc, a4, acc);
                }
            };
            using RF = std::true_type;
            using NR = std::false_type;
            uint32_t t = 0;
            if constexpr (NA == 2u) {
                for (; t + 3u < nc; t += 2) {
                    step(RF{}, t, ra0, ra1, ring);
                    step(RF{}, t + 1u, rb0, rb1, ring + 2048u);
                }
                if (nc - t == 3u) {
                    step(RF{}, t, ra0, ra1, ring);
                    step(NR{}, t + 1u, rb0, rb1, ring + 2048u);
                    step(NR{}, t + 2u, ra0, ra1, ring);
                } else if (nc - t == 2u) {
                    step(NR{}, t, ra0, ra1, ring);
                    step(NR{}, t + 1u, rb0, rb1, ring + 2048u);
                } else if (nc - t == 1u) {
                    step(NR{}, t, ra0, ra1, ring);
                }
            } else {
                for (; t + 5u < nc; t += 3) {
                    step(RF{}, t, ra0, ra1, ring);
                    step(RF{}, t + 1u, rb0, rb1, ring + 2048u);
                    step(RF{}, t + 2u, rc0, rc1, ring + 4096u);
                }
                const uint32_t rem = nc - t;
                if (rem > 3u) {
                    step(RF{}, t, ra0, ra1, ring);
                    if (rem > 4u) step(RF{}, t + 1u, rb0, rb1, ring + 2048u);
                    else step(NR{}, t + 1u, rb0, rb1, ring + 2048u);
                    step(NR{}, t + 2u, rc0, rc1, ring + 4096u);
                    step(NR{}, t + 3u, ra0, ra1, ring);
                    if (rem > 4u) step(NR{}, t + 4u, rb0, rb1, ring + 2048u);
                } else {
                    if (rem > 0u) step(NR{}, t, ra0, ra1, ring);
                    if (rem > 1u) step(NR{}, t + 1u, rb0, rb1, ring + 2048u);
                    if (rem > 2u) step(NR{}, t + 2u, rc0, rc1, ring + 4096u);
                }
            }
            if (g == 0) {
#pragma unroll
                for (int i = 0; i < M; i++) red[slot][part][i][n] = acc[i];
            }
        } else {
            /* the pass's prefetched chunks are not used */
            GHIP_VMCNT(0);
        }
        __syncthreads();
        if (tid < GPP * M * 16u) {
            const uint32_t sl = tid / (M * 16u), rem = tid - sl * (M * 16u);
            const uint32_t m = rem >> 4, nn = rem & 15u;
            const uint32_t gp = ps * GPP + sl;
            if (gp < groups && gp * 16 + nn < O) {
                float s = 0.0f;
#pragma unroll
                for (int k = 0; k < KS; k++) s += red[sl][k][m][nn];
                Y[(size_t)m * O + gp * 16 + nn] = (uint16_t)ghip_bf16_bits(s);
            }
        }
        __syncthreads();
    }
}

static uint32_t g_gs_ncu;                 /* CUs: the streaming grid bound */

/* LDS the streaming GEMV needs for M token rows of length K and `na` chunk
 * slots a wave */
static size_t gs_lds(size_t M, size_t K, size_t na) {
    return ((M * K * 2 + 1023) & ~(size_t)1023) + (size_t)GS_NW * na * 2048;
}

/* FP8: K over two waves, a workgroup per CU; BF16: K over all eight waves, a
 * workgroup per row group. */
template <int M, bool BF>
static hipError_t launch_gemv_m(const void *w, const float *scales, const uint16_t *x, uint16_t *y,
                                size_t O, size_t K, const uint32_t *exact_dev, hipEvent_t ev0,
                                hipEvent_t ev1, hipStream_t st) {
    constexpr int KS = BF ? 8 : 2;
    const size_t groups = (O + 15) / 16;
    const uint32_t grid = BF && groups < g_gs_ncu ? (uint32_t)groups : g_gs_ncu;
    GHIP_LAUNCH(ev0, ev1, (k_fp8_gemv_stream<M, KS, BF>), dim3(grid), dim3(GS_NW * 64),
                gs_lds(M, K, GS_NA(BF)), st, (const uint8_t *)w, scales, x, y, (uint32_t)O,
                (uint32_t)K, exact_dev);
    return hipGetLastError();
}

template <bool BF>
static hipError_t launch_gemv(const void *w, const float *scales, const uint16_t *x, uint16_t *y,
                              size_t M, size_t O, size_t K, const uint32_t *exact_dev,
                              hipEvent_t ev0, hipEvent_t ev1, hipStream_t st) {
    switch (M) {
    case 4: return launch_gemv_m<4, BF>(w, scales, x, y, O, K, exact_dev, ev0, ev1, st);
    case 3: return launch_gemv_m<3, BF>(w, scales, x, y, O, K, exact_dev, ev0, ev1, st);
    case 2: return launch_gemv_m<2, BF>(w, scales, x, y, O, K, exact_dev, ev0, ev1, st);
    default: return launch_gemv_m<1, BF>(w, scales, x, y, O, K, exact_dev, ev0, ev1, st);
    }
}

/* Rows of X from which the MFMA GEMM (N % 256 == 0) is considered. */
#define GHIP_GEMM_MIN_M 16

/* The kernel of an FP8 linear on n_cu CUs. */
extern "C" int ghip_fp8_linear_route(const void *codes, const void *x, const void *y, size_t M,
                                     size_t O, size_t K, uint32_t n_cu) {
    const bool rows = n_cu && ghip_rows_fits(0, M, O, K, codes, x);
    /* up to 4 rows against enough weight rows that every wave holds a row
     * group for half of K: x staged once in LDS (16384 x 4096, M = 1: 11.6 us
     * against 12.0 with x streamed beside the weights; 16384 x 1536: 5.9
     * against 6.2; below that many rows the streamed form is as good or
     * better, 7000 x 2048 4.9 against 6.0) */
    if (rows && M <= 4 && (O + 63) / 64 >= n_cu && M * K * 2 <= GS_X_MAX) return GHIP_ROUTE_GEMV;
    /* below 256 rows whichever is estimated faster, the GEMM where they are
     * within 6% (8192 x 128, M = 100: rows 6.6 us, GEMM 4.6; 1536 x 4096, M =
     * 64: rows 7.7, GEMM 16.5) */
    if (n_cu && n_cu % 8 == 0 && M >= GHIP_GEMM_MIN_M
        && ghip_fp8_gemm_fits(M, O, K, codes, x, y)) {
        if (M >= 256 || !rows) return GHIP_ROUTE_GEMM;
        /* no GEMM is estimated under 4.4 us: the smallest calls skip its plan */
        const float r = 1.06f * ghip_rows_estimate(0, M, O, K, n_cu);
        if (r > 4.4f && ghip_fp8_gemm_estimate(M, O, K, n_cu) < r) return GHIP_ROUTE_GEMM;
    }
    return rows ? GHIP_ROUTE_ROWS : GHIP_ROUTE_ANY;
}

extern "C" hipError_t ghip_launch_fp8_linear(const uint8_t *codes,
                                             const float *scales,
                                             const uint16_t *x, uint16_t *y,
                                             size_t M, size_t O, size_t K,
                                             const uint32_t *exact_dev,
                                             const hipEvent_t *ev,
                                             hipStream_t st) {
    if (M == 0 || O == 0) return hipSuccess;
    if (K == 0 || O > 0x7fffffffu || K > 0x7fffffffu || M > 0x7fffffffu)
        return hipErrorInvalidValue;
    /* timing events: start on the first launch, stop on the last */
    hipEvent_t ev0 = ev ? ev[0] : nullptr, ev1 = ev ? ev[1] : nullptr;
    switch (ghip_fp8_linear_route(codes, x, y, M, O, K, g_gs_ncu)) {
    case GHIP_ROUTE_GEMV:
        return launch_gemv<false>(codes, scales, x, y, M, O, K, exact_dev, ev0, ev1, st);
    case GHIP_ROUTE_GEMM: {
        const hipError_t e =
            ghip_launch_fp8_gemm(codes, scales, x, y, M, O, K, exact_dev, g_gs_ncu, ev, st);
        /* no memory for the K splits, or a capture that would have to allocate
         * it: below 256 rows the form that needs none runs */
        if ((e != hipErrorOutOfMemory && e != hipErrorStreamCaptureUnsupported) || M >= 256
            || !ghip_rows_fits(0, M, O, K, codes, x))
            return e;
        (void)hipGetLastError();
    }
    /* fall through */
    case GHIP_ROUTE_ROWS:
        return ghip_launch_rows(0, codes, scales, x, y, M, O, K, exact_dev, g_gs_ncu, ev0, ev1,
                                st);
    default: return launch_linear_any<false>(codes, scales, x, y, M, O, K, ev0, ev1, st);
    }
}

/* The kernel of a BF16 linear on n_cu CUs. */
extern "C" int ghip_bf16_linear_route(const void *w, const void *x, size_t M, size_t O, size_t K,
                                      uint32_t n_cu) {
    if (!n_cu) return GHIP_ROUTE_ANY;
    const bool rows = ghip_rows_fits(1, M, O, K, w, x);
    /* up to 4 rows against few long weight rows, a chain of chunk round trips
     * with most CUs idle: x staged once and three chunks in flight (288 x 8192,
     * M = 1: 7.1 us against 7.5 with x streamed beside the weights, M = 4 7.5
     * against 7.9; 288 x 4096 4.76 against 4.84, but 288 x 2048 3.63 against
     * 3.56, and 4096 x 4096 7.2 against 7.0) */
    if (rows && M <= 4 && K >= 4096 && O <= 8u * (size_t)n_cu
        && gs_lds(M, K, GS_NA(true)) <= GS_LDS)
        return GHIP_ROUTE_GEMV;
    /* the weight-streaming form reads the weights once per row tile, the
     * GEMM's tiles share them: whichever is estimated faster (4096 x 4096:
     * 12.3 against 15.5 us at M = 64, 20.2 against 15.9 at 96) */
    if (ghip_bf16_gemm_fits(M, O, K, w, x)
        && (!rows || ghip_bf16_gemm_estimate(M, O, K, n_cu) < ghip_rows_estimate(1, M, O, K, n_cu)))
        return GHIP_ROUTE_GEMM;
    return rows ? GHIP_ROUTE_ROWS : GHIP_ROUTE_ANY;
}

extern "C" hipError_t ghip_launch_bf16_linear(const uint16_t *w,
                                              const uint16_t *x, uint16_t *y,
                                              size_t M, size_t O, size_t K,
                                              const hipEvent_t *ev, hipStream_t st) {
    if (M == 0 || O == 0) return hipSuccess;
    if (K == 0 || O > 0x7fffffffu || K > 0x7fffffffu || M > 0x7fffffffu)
        return hipErrorInvalidValue;
    hipEvent_t ev0 = ev ? ev[0] : nullptr, ev1 = ev ? ev[1] : nullptr;
    switch (ghip_bf16_linear_route(w, x, M, O, K, g_gs_ncu)) {
    case GHIP_ROUTE_GEMV:
        return launch_gemv<true>(w, nullptr, x, y, M, O, K, nullptr, ev0, ev1, st);
    case GHIP_ROUTE_GEMM:
        return ghip_launch_bf16_gemm(w, x, y, M, O, K, g_gs_ncu, ev0, ev1, st);
    case GHIP_ROUTE_ROWS:
        return ghip_launch_rows(1, w, nullptr, x, y, M, O, K, nullptr, g_gs_ncu, ev0, ev1, st);
    default: return launch_linear_any<true>(w, nullptr, x, y, M, O, K, ev0, ev1, st);
    }
}

extern "C" hipError_t ghip_linear_init(uint32_t n_cu) {
    const void *ks[8] = {
        (const void *)k_fp8_gemv_stream<1, 2, false>, (const void *)k_fp8_gemv_stream<2, 2, false>,
        (const void *)k_fp8_gemv_stream<3, 2, false>, (const void *)k_fp8_gemv_stream<4, 2, false>,
        (const void *)k_fp8_gemv_stream<1, 8, true>, (const void *)k_fp8_gemv_stream<2, 8, true>,
        (const void *)k_fp8_gemv_stream<3, 8, true>, (const void *)k_fp8_gemv_stream<4, 8, true>};
    hipError_t e;
    for (int i = 0; i < 8; i++)
        if ((e = hipFuncSetAttribute(ks[i], hipFuncAttributeMaxDynamicSharedMemorySize, GS_LDS))
            != hipSuccess)
            return e;
    if ((e = ghip_rows_init()) != hipSuccess) return e;
    if ((e = ghip_bf16_gemm_init()) != hipSuccess) return e;
    g_gs_ncu = n_cu;
    return hipSuccess;
}
