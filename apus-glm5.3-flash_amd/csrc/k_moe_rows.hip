/*
 * k_moe_rows.hip — routed-MoE prefill for few tokens (gfx950): the gate/up +
 * SwiGLU and down products of expert tiles that mostly hold a few rows, as
 * weight streams (c/gmoe.h:210-227 per token in the reference).
 *
 * An item is rows of one tile of the expert-sorted rows (k_moe_prefill.hip) against
 * 16 gate and the same 16 up rows (MODE 0) or 64 down rows (MODE 1), 128 KB of
 * weights at dim 4096 / inter 2048. The 8 waves split K (8 ways, or 4 ways
 * over two groups of 32 down rows); a wave loads 128-wide k blocks of its 32
 * weight rows with that part of 16 activation rows (gathered by token in MODE
 * 0) into registers, passes both through a wave-private LDS area into the
 * layout of v_mfma_f32_16x16x32_bf16 and dequantizes each code once. The
 * partial sums meet in LDS in a fixed order. An item takes up to 32 rows, in
 * passes of 16 (the weights come from L2 again); a tile's further rows are
 * items of their own.
 *
 * HBM bounds it: 6.2-6.3 TB/s at T = 12, top-8 of 288 (1.39 GB of gate/up in
 * 224 us, 0.69 GB of down in 110; by the counters the bytes fetched are the
 * weights' and the matrix cores are busy 9% of the cycles). Two workgroups a CU (64 KB of LDS, 128
 * registers a lane) keep loads in flight across items, and small items keep
 * all CUs busy from the first token on, where the tile GEMM's 1 MB items and
 * ~25 us a launch do not: T = 2 135 -> 79 us, T = 12 426 -> 345, 16 experts
 * of 1024/512 at T = 16 66 -> 20.
 */
#include "ghip_device.h"
#include "ghip_internal.h"

#define MR_NW 8
#define MR_SLOT (4096u + 4096u)  /* x of 16 rows, two weight chunks */
#define MR_LDS (MR_NW * MR_SLOT)
#define MR_SUB ((uint32_t)PF_LONG_ROWS)  /* rows of an item */
#define MR_LONG 512u             /* most tiles of more rows */

/* One item for `rows` (1..16) sorted rows from row0. */
template <int MODE, bool EXACT>
__device__ __forceinline__ void mr_body(const GhipBank &bank, const uint16_t *__restrict__ act,
                                        const int32_t *__restrict__ perm, uint32_t e,
                                        uint32_t row0, uint32_t rows, uint32_t nb, uint32_t topk,
                                        float limit, uint16_t *__restrict__ out, uint8_t *lds) {
    constexpr uint32_t KS = MODE == 0 ? 8u : 4u;         /* K splits */
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t n = lane & 15u, g = lane >> 4;
    const uint32_t part = wv % KS, slot = wv / KS;
    const uint32_t K = MODE == 0 ? bank.dim : bank.inter;
    const uint32_t nch = K >> 7;
    const uint32_t c0 = part * nch / KS, nc = (part + 1u) * nch / KS - c0;
    const uint8_t *slab = bank.base + (size_t)e * bank.stride;
    /* weight rows: 16 gate and 16 up rows (MODE 0), 32 down rows (MODE 1) */
    const uint32_t wr0 = MODE == 0 ? nb * 16u : nb * 64u + slot * 32u;
    const uint8_t *w0 = slab + (MODE == 0 ? bank.off_gw : bank.off_dw) + (size_t)wr0 * K;
    const uint8_t *w1 = MODE == 0 ? slab + bank.off_uw + (size_t)wr0 * K : w0 + (size_t)16u * K;
    const float *s0 = (const float *)(slab + (MODE == 0 ? bank.off_gs : bank.off_ds))
                    + (size_t)(wr0 >> 7) * nch;
    const float *s1 = MODE == 0 ? (const float *)(slab + bank.off_us) + (size_t)(wr0 >> 7) * nch : s0;
    uint8_t *xs = lds + wv * MR_SLOT, *ws = xs + 4096u;
    ghip_f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
    const ghip_cdma d = ghip_cdma_offsets(lane, K);
    /* x load u: rows 4u + l / 16, piece l % 16 of the row's 256 bytes */
    uint32_t xo[4];
#pragma unroll
    for (uint32_t u = 0; u < 4; u++) {
        const uint32_t r = 4u * u + (lane >> 4), rc = row0 + min(r, rows - 1u);
        const uint32_t src = MODE == 0 ? (uint32_t)perm[rc] / topk : rc;
        xo[u] = src * K * 2u + 16u * ((lane & 15u) ^ (r & 15u));
    }
    ghip_u32x4 xr[4], a0, a1, b0, b1;
    float sa, sb;
    /* the scales as vector loads, in order with the codes: a scalar load would
     * make every LDS wait of the step wait for it */
    auto load = [&](uint32_t c) {
        const uint8_t *xc = (const uint8_t *)act + (size_t)c * 256u;
#pragma unroll
        for (uint32_t u = 0; u < 4; u++) xr[u] = *(const ghip_u32x4 *)(xc + xo[u]);
        ghip_rl_load(w0, d, c, a0, a1);
        ghip_rl_load(w1, d, c, b0, b1);
        sa = __uint_as_float(__hip_atomic_load((const uint32_t *)s0 + c, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_WORKGROUP));
        sb = MODE == 0 ? __uint_as_float(__hip_atomic_load((const uint32_t *)s1 + c, __ATOMIC_RELAXED,
                                                           __HIP_MEMORY_SCOPE_WORKGROUP))
                       : sa;
        __builtin_amdgcn_sched_barrier(0);
    };
    if (nc) load(c0);
    for (uint32_t t = 0; t < nc; t++) {
#pragma unroll
        for (uint32_t u = 0; u < 4; u++) *(ghip_u32x4 *)(xs + u * 1024u + lane * 16u) = xr[u];
        ghip_rl_store(ws, lane, a0, a1);
        ghip_rl_store(ws + 2048u, lane, b0, b1);
        const float fa = sa, fb = sb;
        __builtin_amdgcn_sched_barrier(0);
        if (t + 1u < nc) load(c0 + t + 1u);
        __builtin_amdgcn_sched_barrier(0);
        const ghip_chunk ca = ghip_cdma_read(ws, n, g), cb = ghip_cdma_read(ws + 2048u, n, g);
        ghip_bf16x8 wa[4], wb[4];
        ghip_deq16<EXACT>(ca.lo, fa, wa[0], wa[1]);
        ghip_deq16<EXACT>(ca.hi, fa, wa[2], wa[3]);
        ghip_deq16<EXACT>(cb.lo, fb, wb[0], wb[1]);
        ghip_deq16<EXACT>(cb.hi, fb, wb[2], wb[3]);
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) {
            const ghip_bf16x8 xv = *(const ghip_bf16x8 *)(xs + n * 256u + 16u * ((4u * g + i) ^ n));
            acc0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xv, wa[i], acc0, 0, 0, 0);
            acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xv, wb[i], acc1, 0, 0, 0);
        }
    }
    __syncthreads();
    float *red = (float *)lds;                           /* [8 waves][16 rows][32] */
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) {
        red[(wv * 16u + 4u * g + i) * 32u + n] = acc0[i];
        red[(wv * 16u + 4u * g + i) * 32u + 16u + n] = acc1[i];
    }
    __syncthreads();
    if constexpr (MODE == 0) {
        const uint32_t m = tid >> 4, c = tid & 15u;      /* 16 rows x 16 columns (tid < 256) */
        if (m < 16u && m < rows) {
            float gs = 0.0f, us = 0.0f;
#pragma unroll
            for (uint32_t k = 0; k < KS; k++) {
                gs += red[(k * 16u + m) * 32u + c];
                us += red[(k * 16u + m) * 32u + 16u + c];
            }
            out[(size_t)(row0 + m) * bank.inter + wr0 + c] =
                (uint16_t)ghip_swiglu(ghip_bf16_round(gs), ghip_bf16_round(us), limit);
        }
    } else {
#pragma unroll
        for (uint32_t v = tid; v < 16u * 64u; v += MR_NW * 64u) {
            const uint32_t m = v >> 6, c = v & 63u, sl = c >> 5, cc = c & 31u;
            if (m < rows) {
                float s = 0.0f;
#pragma unroll
                for (uint32_t k = 0; k < KS; k++)
                    s += red[((sl * KS + k) * 16u + m) * 32u + cc];
                out[(size_t)(row0 + m) * bank.dim + nb * 64u + c] = (uint16_t)ghip_bf16_bits(s);
            }
        }
    }
    __syncthreads();
}

/* Persistent, two workgroups a CU, items dealt round-robin. An item is MR_SUB
 * rows at most: a tile's rows past that are items of their own, after the
 * others', from a list of the longer tiles that every workgroup makes (so one
 * expert with most of the rows keeps all CUs busy and not a few with 16
 * passes each: 128 experts of 512/256, top-2, Zipf 1.1, T = 600 93 -> 51 us,
 * T = 1500 110 -> 67; parts of 64 rows 58 and 73). An
 * item's parts keep its column block, hence its XCD where nblk % 8 == 0. */
template <int MODE>
__global__ __launch_bounds__(MR_NW * 64, 4) void k_moe_rows(
    GhipBank bank, const uint16_t *__restrict__ act, const int32_t *__restrict__ perm,
    const uint4 *__restrict__ tiles, const uint32_t *__restrict__ hdr, uint32_t topk, float limit,
    uint16_t *__restrict__ out) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t mr_lds[];
    uint16_t *longer = (uint16_t *)(mr_lds + MR_LDS);    /* tiles of more than MR_SUB rows */
    const uint32_t nblk = MODE == 0 ? bank.inter / 16u : bank.dim / 64u;
    const uint32_t ntiles = hdr[PF_HDR_NTILES], items = ntiles * nblk;
    uint32_t nlong = 0;
    if (hdr[PF_HDR_LONG]) {
        uint32_t *cnt = (uint32_t *)mr_lds;
        const uint32_t tid = threadIdx.x, w = tid >> 6;
        for (uint32_t t0 = 0; t0 < ntiles; t0 += MR_NW * 64u) {
            const bool is = t0 + tid < ntiles && tiles[t0 + tid].z > MR_SUB;
            const uint64_t m = __ballot(is);
            if ((tid & 63u) == 0) cnt[w] = __popcll(m);
            __syncthreads();
            uint32_t at = nlong + __popcll(m & ((1ull << (tid & 63u)) - 1ull));
            for (uint32_t v = 0; v < MR_NW; v++) {
                if (v < w) at += cnt[v];
                nlong += cnt[v];
            }
            if (is && at < MR_LONG) longer[at] = (uint16_t)(t0 + tid);
            __syncthreads();
        }
        nlong = __builtin_amdgcn_readfirstlane(min(nlong, MR_LONG));
    }
    const uint32_t total = items + nlong * nblk * (PF_BM / MR_SUB - 1u);
    for (uint32_t it = blockIdx.x; it < total; it += gridDim.x) {
        uint32_t ti = it / nblk, from = 0;
        const uint32_t nb = it - ti * nblk;
        if (it >= items) {
            const uint32_t j = ti - ntiles;              /* q-major: part 1 of every tile first */
            const uint32_t q = j / nlong;
            ti = __builtin_amdgcn_readfirstlane(longer[j - q * nlong]);
            from = (q + 1u) * MR_SUB;
        }
        const uint4 td = tiles[ti];
        const uint32_t end = min(td.z, from + MR_SUB);
        for (uint32_t m0 = from; m0 < end; m0 += 16u) {
            const uint32_t rows = min(end - m0, 16u), r0 = td.y + m0;
            if (td.w & 1u)
                mr_body<MODE, true>(bank, act, perm, td.x, r0, rows, nb, topk, limit, out, mr_lds);
            else
                mr_body<MODE, false>(bank, act, perm, td.x, r0, rows, nb, topk, limit, out, mr_lds);
        }
    }
}

/* 32-bit activation offsets, and MR_LONG tiles of over MR_SUB rows at most */
extern "C" int ghip_moe_rows_fits(uint32_t dim, uint32_t inter, size_t T, size_t P) {
    return dim % 128 == 0 && inter % 128 == 0 && P <= (size_t)MR_LONG * MR_SUB
        && T * dim * 2 <= 0xffffffffull && P * inter * 2 <= 0xffffffffull;
}

extern "C" hipError_t ghip_launch_moe_rows(int mode, const GhipBank *bank, const uint16_t *act,
                                           const int32_t *perm, const uint32_t *tiles,
                                           const uint32_t *hdr, uint32_t topk, float limit,
                                           uint16_t *out, uint32_t n_cu, hipEvent_t e0,
                                           hipEvent_t e1, hipStream_t st) {
    if (!bank || !act || !perm || !tiles || !hdr || !out || n_cu == 0 || bank->dim % 128
        || bank->inter % 128 || bank->inter == 0 || bank->dim == 0)
        return hipErrorInvalidValue;
    const dim3 grid(2u * n_cu), blk(MR_NW * 64);
    if (mode == 0)
        GHIP_LAUNCH(e0, e1, k_moe_rows<0>, grid, blk, MR_LDS + MR_LONG * 2u, st, *bank, act, perm,
                    (const uint4 *)tiles, hdr, topk, limit, out);
    else
        GHIP_LAUNCH(e0, e1, k_moe_rows<1>, grid, blk, MR_LDS + MR_LONG * 2u, st, *bank, act, perm,
                    (const uint4 *)tiles, hdr, topk, limit, out);
    return hipGetLastError();
}

extern "C" hipError_t ghip_moe_rows_init(void) {
    const void *ks[2] = {(const void *)k_moe_rows<0>, (const void *)k_moe_rows<1>};
    for (int i = 0; i < 2; i++) {
        hipError_t e = hipFuncSetAttribute(ks[i], hipFuncAttributeMaxDynamicSharedMemorySize,
                                           MR_LDS + MR_LONG * 2);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
