/*
 * k_dequant.hip — K1, FP8-E4M3 + F32 128x128 scales -> BF16, bit-exact vs
 * c/fp8blk.h:115-136 (apus_fp8blk_rows_scalar).
 */
#include "ghip_device.h"
#include "ghip_internal.h"

#define DQ_CHUNK 8u              /* codes a lane takes at a time: stores of 16 bytes */
#define DQ_U 2u                  /* chunks in flight a lane */

/* Eight codes (two dwords) with one scale each -> 16 bytes of bf16. EXACT:
 * the hardware convert with the NaN codes replaced gives the reference's bits
 * for every finite scale; a product with a scale that is not finite may be a
 * NaN, whose bits only the integer narrow passes through. */
template <bool EXACT, bool ANYK>
__device__ __forceinline__ ghip_u32x4 dq_eight(uint2 c, const float (&s)[3], uint32_t e0,
                                               uint32_t e1) {
    typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
    bool finite = true;
    if (EXACT) {
        finite = __builtin_fabsf(s[0]) < __builtin_inff();
        if (ANYK)
            finite = finite && __builtin_fabsf(s[1]) < __builtin_inff()
                     && __builtin_fabsf(s[2]) < __builtin_inff();
    }
    auto scale = [&](uint32_t j) {
        return !ANYK ? s[0] : j < e0 ? s[0] : j < e1 ? s[1] : s[2];
    };
    ghip_u32x4 r;
    if (finite) {
#pragma unroll
        for (uint32_t h = 0; h < 4; h++) {
            const uint32_t d = h < 2 ? c.x : c.y;
            ghip_f32x2 v = h & 1u ? __builtin_amdgcn_cvt_pk_f32_fp8((int)d, true)
                                  : __builtin_amdgcn_cvt_pk_f32_fp8((int)d, false);
            if (EXACT) {
                v[0] = ghip_e4m3_fix(v[0], h & 1u ? d << 8 : d << 24);
                v[1] = ghip_e4m3_fix(v[1], h & 1u ? d : d << 16);
            }
            bf2 p;
            p[0] = (__bf16)(v[0] * scale(2u * h));
            p[1] = (__bf16)(v[1] * scale(2u * h + 1u));
            r[h] = __builtin_bit_cast(uint32_t, p);
        }
    } else {
#pragma unroll
        for (uint32_t h = 0; h < 4; h++) {
            const uint32_t d = (h < 2 ? c.x : c.y) >> (16u * (h & 1u));
            const uint32_t lo = ghip_bf16_bits(ghip_e4m3_exact(d & 0xffu) * scale(2u * h));
            const uint32_t hi = ghip_bf16_bits(ghip_e4m3_exact((d >> 8) & 0xffu)
                                               * scale(2u * h + 1u));
            r[h] = lo | (hi << 16);
        }
    }
    return r;
}

/* Bound by HBM: 1 byte read and 2 written a code, 16384 x 4096 29.2 us, 6.9
 * TB/s (a device copy of 200 MB: 5.4). What it took: whole lines per store
 * instruction (a lane's 16 codes as two stores of stride 32, with the integer
 * decode's ~20 operations a code: 42.9 us; this form with ordinary stores
 * 37.5), stores that pass the caches (29.2), and two chunks a lane (one 31.2,
 * four 29.8, and 4.0 against 3.5 us at 2048 x 2048). A width that is no
 * multiple of 8, 16384 x 1999, takes 16.1 us.
 *
 * The matrix is one run of O * K codes in chunks of 8; a workgroup takes
 * DQ_U x 256 consecutive chunks. The one division by K of 64 bits is uniform, the
 * lanes' are of 32 bits. K % 8 == 0 (!ANYK): a chunk has one scale. ANYK (K
 * >= 8): a chunk meets at most one end of a scale block and one end of a row,
 * so it has up to three scales, up to element e0, e1 and the end; the last
 * chunk may be partial. */
template <bool EXACT, bool ANYK>
__global__ __launch_bounds__(256) void k_dequant(
    const uint8_t *__restrict__ w, const float *__restrict__ s,
    uint16_t *__restrict__ out, uint32_t O, uint32_t K, uint32_t nkb) {
    const size_t n = (size_t)O * K, nc = n / DQ_CHUNK;
    const size_t c0 = (size_t)blockIdx.x * (DQ_U * 256u);
    const uint32_t left = (uint32_t)min((size_t)(DQ_U * 256u), nc - min(c0, nc));
    const size_t i0 = c0 * DQ_CHUNK;
    const uint32_t row0 = (uint32_t)(i0 / K), k0 = (uint32_t)(i0 - (size_t)row0 * K);
    uint2 c[DQ_U];
    float sc[DQ_U][3];
    uint32_t e0[DQ_U], e1[DQ_U];
#pragma unroll
    for (uint32_t u = 0; u < DQ_U; u++) {
        const uint32_t t = u * 256u + threadIdx.x;
        if (t >= left) continue;
        c[u] = *(const uint2 *)(w + i0 + t * DQ_CHUNK);
        const uint32_t a = k0 + t * DQ_CHUNK, dr = a / K, k = a - dr * K, row = row0 + dr;
        const float *sr = s + (size_t)(row >> 7) * nkb;
        sc[u][0] = sr[k >> 7];
        if (ANYK) {
            const uint32_t blk = 128u - (k & 127u), end = K - k;
            e0[u] = min(blk, end);
            e1[u] = end;
            sc[u][1] = sr[min((k >> 7) + 1u, nkb - 1u)];
            sc[u][2] = s[(size_t)(min(row + 1u, O - 1u) >> 7) * nkb];
        }
    }
#pragma unroll
    for (uint32_t u = 0; u < DQ_U; u++) {
        const uint32_t t = u * 256u + threadIdx.x;
        if (t >= left) continue;
        const ghip_u32x4 r = dq_eight<EXACT, ANYK>(c[u], sc[u], e0[u], e1[u]);
        __builtin_nontemporal_store(r, (ghip_u32x4 *)(out + i0 + t * DQ_CHUNK));
    }
    if (ANYK && blockIdx.x == gridDim.x - 1u && threadIdx.x < (uint32_t)(n - nc * DQ_CHUNK)) {
        /* fewer than 8 codes, all of the last row (K >= 8) */
        const size_t i = nc * DQ_CHUNK + threadIdx.x;
        const uint32_t k = (uint32_t)(i - (size_t)(O - 1u) * K);
        out[i] = (uint16_t)ghip_bf16_bits(
            ghip_e4m3_exact(w[i]) * s[(size_t)((O - 1u) >> 7) * nkb + (k >> 7)]);
    }
}

/* Any K, any alignment: one thread per element, exact integer path. */
__global__ __launch_bounds__(256) void k_dequant_any(
    const uint8_t *__restrict__ w, const float *__restrict__ s,
    uint16_t *__restrict__ out, uint32_t O, uint32_t K, uint32_t nkb) {
    const size_t n = (size_t)O * K;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n;
         i += (size_t)gridDim.x * 256) {
        uint32_t o = (uint32_t)(i / K), k = (uint32_t)(i - (size_t)o * K);
        float sc = s[(size_t)(o >> 7) * nkb + (k >> 7)];
        out[i] = (uint16_t)ghip_bf16_bits(ghip_e4m3_exact(w[i]) * sc);
    }
}

extern "C" size_t ghip_dequant_rows(size_t O, size_t K) {
    const size_t most = GHIP_MAX_THREADS / 256u * (DQ_U * 256u * DQ_CHUNK);
    return O <= most / K ? O : most / K / 128u * 128u;
}

extern "C" hipError_t ghip_launch_dequant(const uint8_t *codes,
                                          const float *scales, uint16_t *out,
                                          size_t O, size_t K, int exact,
                                          hipStream_t st) {
    if (O == 0 || K == 0) return hipSuccess;
    if (O > 0xffffffffu || K > 0xffffffffu) return hipErrorInvalidValue;
    const uint32_t nkb = (uint32_t)((K + 127) / 128);
    const size_t per = DQ_U * 256u * DQ_CHUNK, rows = ghip_dequant_rows(O, K);
    /* rows of under 8 codes could end twice in a chunk; the sums of a
     * workgroup's k and of its blocks stay within 32 bits */
    if (K >= DQ_CHUNK && K <= 0x7fffffffu && rows && ((uintptr_t)codes & 7) == 0
        && ((uintptr_t)out & 15) == 0) {
        for (size_t r = 0; r < O; r += rows) {
            const size_t n = O - r < rows ? O - r : rows;
            const dim3 g((uint32_t)((n * K + per - 1) / per));
            const uint8_t *w = codes + r * K;
            const float *s = scales + (r / 128) * nkb;
            uint16_t *o = out + r * K;
            /* the fast decode is for K % 16 == 0 and 16-byte aligned codes only:
             * elsewhere NaN codes have their numbers whatever `exact` says */
            if (K % 8)
                hipLaunchKernelGGL((k_dequant<true, true>), g, dim3(256), 0, st, w, s, o,
                                   (uint32_t)n, (uint32_t)K, nkb);
            else if (exact || K % 16 || ((uintptr_t)codes & 15))
                hipLaunchKernelGGL((k_dequant<true, false>), g, dim3(256), 0, st, w, s, o,
                                   (uint32_t)n, (uint32_t)K, nkb);
            else
                hipLaunchKernelGGL((k_dequant<false, false>), g, dim3(256), 0, st, w, s, o,
                                   (uint32_t)n, (uint32_t)K, nkb);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    size_t g = (O * K + 255) / 256;
    if (g > 65536) g = 65536;
    hipLaunchKernelGGL(k_dequant_any, dim3((uint32_t)g), dim3(256), 0, st, codes,
                       scales, out, (uint32_t)O, (uint32_t)K, nkb);
    return hipGetLastError();
}
