"""Which kernel a linear or a prefill takes (csrc/k_linear.hip,
csrc/k_moe_prefill.hip), asked of the library's own dispatch: host code, so no
device and no buffers of these sizes are needed."""
import ctypes
import random

import pytest

ANY, GEMV, ROWS, GEMM = range(4)
NCU = 256
P = ctypes.c_void_p(1 << 20)


def fp8(pkg, M, N, K, codes=P, x=P, y=P, ncu=NCU):
    f = pkg.load().ghip_fp8_linear_route
    f.restype = ctypes.c_int
    f.argtypes = [ctypes.c_void_p] * 3 + [ctypes.c_size_t] * 3 + [ctypes.c_uint32]
    return f(codes, x, y, M, N, K, ncu)


# the most rows that 65535 row tiles of 16 rows hold, and more than 65535
# tiles of any height
EDGE = 65535 * 16


@pytest.mark.parametrize("M", [EDGE, EDGE + 1, 1300000])
def test_fp8_very_many_rows_stay_on_the_gemm(pkg, M):
    """What the MFMA GEMM takes (N % 256 == 0, 2 M K under 4 GiB) goes there
    at any number of rows."""
    assert fp8(pkg, M, 16384, 1536) == GEMM
    assert fp8(pkg, M, 256, 128) == GEMM


@pytest.mark.parametrize("M", [EDGE, EDGE + 1, 65535 * 64 + 1, 0x7FFFFFFF])
def test_fp8_very_many_rows_off_the_gemm(pkg, M):
    """What it does not take is streamed, in as many launches as its row tiles
    need, and never falls to the kernel of any shape."""
    assert fp8(pkg, M, 300, 128) == ROWS
    assert fp8(pkg, M, 16384, 4096) == ROWS          # 2 M K over 4 GiB


def test_fp8_other_shapes(pkg):
    off = ctypes.c_void_p(P.value + 2)
    assert fp8(pkg, 1, 16384, 4096) == GEMV and fp8(pkg, 4, 16384, 1536) == GEMV
    assert fp8(pkg, 5, 16384, 4096) == ROWS and fp8(pkg, 1, 512, 4096) == ROWS
    assert fp8(pkg, 256, 512, 4096) == GEMM and fp8(pkg, 256, 500, 4096) == ROWS
    assert fp8(pkg, 1, 512, 4095) == ANY and fp8(pkg, 300, 512, 4096, codes=off) == ANY
    assert fp8(pkg, 300, 512, 4096, x=off) == ANY and fp8(pkg, 300, 512, 4096, y=off) == ROWS
    assert fp8(pkg, 300, 512, 4096, ncu=0) == ANY


@pytest.mark.parametrize("O,K", [(1, 128), (16384, 4096), (1 << 24, 4096), ((1 << 24) - 1, 4096), (1 << 25, 4096),
                                 (1 << 32, 16), (9000000, 8191), (130, 1 << 29), (130, (1 << 29) + 8)])
def test_dequant_launches_stay_under_the_thread_limit(pkg, O, K):
    """The rows of one launch: whole scale blocks, 2^32 threads or more in
    none (8 codes a thread, 512 chunks of 8 a workgroup of 256)."""
    f = pkg.load().ghip_dequant_rows
    f.restype, f.argtypes = ctypes.c_size_t, [ctypes.c_size_t] * 2
    rows = f(O, K)
    assert rows == O or rows % 128 == 0
    assert (rows * K + 4095) // 4096 * 256 < 1 << 32
    # as many as fit: twice the rows (or a block more) would not
    assert rows == O or ((rows + 128) * K + 4095) // 4096 * 256 >= 1 << 32


# (M, N, K), the faster kernel, by a tenth or more (measured on 256 CUs)
FEW = [(100, 8192, 128, GEMM), (255, 12288, 128, GEMM), (160, 12288, 512, GEMM), (96, 16384, 256, GEMM),
       (64, 32768, 256, GEMM), (255, 8192, 768, GEMM), (128, 16384, 1536, GEMM), (17, 32768, 128, GEMM),
       (16, 16384, 1536, ROWS), (64, 1536, 4096, ROWS), (129, 1536, 4096, ROWS), (64, 512, 4096, ROWS),
       (32, 16384, 4096, ROWS), (48, 2048, 2048, ROWS)]


@pytest.mark.parametrize("M,N,K,want", FEW)
def test_fp8_few_rows_take_the_faster_kernel(pkg, M, N, K, want):
    assert fp8(pkg, M, N, K) == want


def bf16(pkg, M, N, K, w=P, x=P, ncu=NCU):
    f = pkg.load().ghip_bf16_linear_route
    f.restype, f.argtypes = ctypes.c_int, [ctypes.c_void_p] * 2 + [ctypes.c_size_t] * 3 + [ctypes.c_uint32]
    return f(w, x, M, N, K, ncu)


def test_bf16_routes(pkg):
    off = ctypes.c_void_p(P.value + 2)
    # few long weight rows: x staged once
    assert all(bf16(pkg, M, N, K) == GEMV for M in (1, 2, 4) for N in (64, 288, 2048) for K in (4096, 8192))
    assert bf16(pkg, 1, 288, 2048) == ROWS and bf16(pkg, 1, 4096, 4096) == ROWS and bf16(pkg, 5, 288, 8192) == ROWS
    assert bf16(pkg, 4, 288, 12288) == GEMV and bf16(pkg, 4, 288, 12288 + 64) == ROWS    # x in LDS
    assert bf16(pkg, 1, 154880, 4096) == ROWS and bf16(pkg, 600, 4096, 4096) == GEMM
    assert bf16(pkg, 2048, 288, 4096) == GEMM and bf16(pkg, 65535 * 64 + 1, 48, 64) in (ROWS, GEMM)
    assert bf16(pkg, 1, 288, 4095) == ANY and bf16(pkg, 1, 288, 4096, w=off) == ANY
    assert bf16(pkg, 1, 288, 4096, x=off) == ANY and bf16(pkg, 1, 288, 4096, ncu=0) == ANY


def test_every_form_that_is_picked_has_a_gpu_case(pkg):
    """The forms of the streaming kernel, the tiles of the BF16 GEMM and the
    heights of the FP8 one that shapes drawn at random reach are those that
    the GPU tests hold a case to."""
    import test_gpu_bf16_gemm
    import test_gpu_fp8_gemm
    import test_gpu_rows
    lib, rng, z = pkg.load(), random.Random(2), ctypes.c_size_t
    seen = {ROWS: set(), "bf16": set(), GEMM: set(), "fp8": set()}
    for _ in range(20000):
        M, N = int(2 ** rng.uniform(0, 11.5)), int(2 ** rng.uniform(4, 17))
        K = 128 * int(2 ** rng.uniform(0, 7.1))
        if rng.random() < 0.5:
            N = N // 256 * 256 + 256
        r = fp8(pkg, M, N, K)
        if r == ROWS:
            f = lib.ghip_rows_form(0, z(M), z(N), z(K), NCU)
            seen[ROWS].add((f >> 16, f >> 8 & 255, f & 255))
        elif r == GEMM:
            f = lib.ghip_fp8_gemm_form(z(M), z(N), z(K), NCU)
            seen["fp8"].add((f >> 16, (f & 0xffff) > 1))
        r = bf16(pkg, M, N, K // 2)
        if r == ROWS:
            f = lib.ghip_rows_form(1, z(M), z(N), z(K // 2), NCU)
            seen["bf16"].add((f >> 16, f >> 8 & 255, f & 255))
        elif r == GEMM:
            f = lib.ghip_bf16_gemm_form(z(M), z(N), NCU)
            seen[GEMM].add((f >> 16, f & 0xffff))
    assert seen[ROWS] <= set(test_gpu_rows.FP8.values())
    assert seen["bf16"] <= set(test_gpu_rows.BF16.values())
    assert seen[GEMM] <= set(test_gpu_bf16_gemm.SHAPES.values())
    assert seen["fp8"] <= {(h, s > 1) for h, s in test_gpu_fp8_gemm.SHAPES.values()}


QUEUED, FULL, STREAMS = range(3)


@pytest.mark.parametrize("dim,inter,experts,k,T,want", [
    (4096, 2048, 288, 8, 12, STREAMS), (4096, 2048, 288, 8, 31, STREAMS), (4096, 2048, 289, 9, 28, STREAMS),
    (4096, 2048, 288, 8, 64, QUEUED),
    (4096, 2048, 288, 8, 4608, FULL), (64 * 32, 1024, 65, 7, 32, STREAMS), (512, 256, 128, 2, 1500, STREAMS),
    # about one row an expert on average; the second: half a row, but 20 experts' weights where all tokens
    # choose the same ones
    (4096, 2048, 288, 8, 36, QUEUED), (4096, 2048, 600, 4, 75, QUEUED), (4096, 2048, 289, 9, 32, QUEUED)])
def test_prefill_form(pkg, dim, inter, experts, k, T, want):
    f = pkg.load().ghip_moe_prefill_form
    f.argtypes = [ctypes.c_uint32] * 4 + [ctypes.c_size_t]
    assert f(dim, inter, experts, k, T) == want


@pytest.mark.parametrize("dim,inter,k,T", [
    (4096, 2048, 8, 8192), (4096, 2048, 8, 131071), (4096, 2048, 8, 131072), (4096, 2048, 9, 1 << 20), (256, 16384, 1, 131272),
    (16384, 128, 1, 131071), (16384, 128, 1, 131072), (256, 128, 1, 1 << 25), (256, 128, 16, 1)])
def test_prefill_slices_keep_offsets_in_32_bits(pkg, dim, inter, k, T):
    f = pkg.load().ghip_moe_prefill_tokens
    f.restype, f.argtypes = ctypes.c_size_t, [ctypes.c_uint32] * 3 + [ctypes.c_size_t]
    n = f(dim, inter, k, T)
    assert 1 <= n <= T and n * dim * 2 < 1 << 32 and n * k * inter * 2 < 1 << 32
    fits = T * dim * 2 < 1 << 32 and T * k * inter * 2 < 1 << 32
    assert (n == T) == fits
