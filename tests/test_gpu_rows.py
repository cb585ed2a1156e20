"""The weight-streaming linear for a few rows (csrc/k_rows.hip) behind the
fp8blk_linear and bf16_gemm entries, against the oracle to the contract
tolerance (tests/tolerance.py): each form the launcher picks (rows of x,
weight groups, K splits), fewer chunks than waves, odd chunk counts, row and
column remainders, x too large to stage, NaN codes by the exact decode, and a
result two bytes off a 16-byte boundary."""
import ctypes

import numpy as np
import pytest

import oracle as O
import gpu_util as G
from tolerance import assert_close

pytestmark = pytest.mark.gpu

# (M, N, K): the form the library picks on 256 CUs as rows of x, weight groups, K splits, to which each case is held
FP8 = {(1, 100, 128): (4, 1, 8), (2, 33, 256): (4, 1, 8), (4, 1000, 1152): (4, 1, 8),    # one chunk; 9 chunks
       (3, 4096, 16384): (4, 1, 8),                                                    # x over 48 KB
       (3, 9001, 384): (4, 1, 4), (4, 6000, 512): (4, 1, 4), (1, 8551, 128): (4, 1, 2),
       (7, 1000, 1024): (8, 1, 8), (5, 4285, 384): (8, 1, 4), (8, 15000, 384): (8, 1, 2), (5, 9000, 640): (8, 1, 2),
       (17, 1000, 896): (16, 1, 8), (16, 7000, 1024): (16, 2, 8), (50, 2000, 1024): (16, 2, 8),
       (13, 16383, 512): (16, 2, 4), (300, 500, 256): (16, 2, 4),
       (1040, 99, 640): (32, 1, 8), (17, 4115, 640): (32, 2, 8), (24, 16383, 384): (32, 2, 4),
       (33, 7000, 640): (32, 2, 4), (64, 16380, 384): (32, 2, 4), (65, 16001, 128): (32, 2, 4),
       (33, 24854, 128): (64, 2, 4), (67, 7582, 640): (64, 2, 4), (100, 5569, 640): (64, 2, 4)}
BF16 = {(1, 288, 1024): (8, 1, 8), (8, 500, 64): (8, 1, 8), (3, 20000, 192): (8, 1, 4),
        (9, 300, 128): (16, 1, 8), (30, 2000, 576): (16, 1, 8), (17, 2188, 64): (16, 1, 4),
        (40, 2100, 64): (16, 1, 4), (12, 8200, 512): (16, 2, 4), (16, 20000, 256): (16, 2, 4),
        (60, 2000, 1024): (32, 1, 8), (17, 4140, 320): (32, 2, 8), (33, 4000, 320): (32, 2, 8),
        (17, 8417, 128): (32, 2, 4), (31, 9000, 192): (32, 2, 4)}
ROWS = 2                                                            # the route's number (ghip_internal.h)


def held_to_form(ghip, bf, M, N, K, form):
    """The dispatch's choices are host code over estimates: a changed one must
    not take a form's cases away unseen."""
    p, z = ctypes.c_void_p(1 << 20), [ctypes.c_size_t(v) for v in (M, N, K)]
    route = ghip.ghip_bf16_linear_route(p, p, *z, 256) if bf else ghip.ghip_fp8_linear_route(p, p, p, *z, 256)
    got = ghip.ghip_rows_form(bf, *z, 256)
    assert route == ROWS and (got >> 16, got >> 8 & 255, got & 255) == form


def guarded(ghip, call, M, N, pad):
    guard = np.full(M * N + 64, 0x7E57, np.uint16)
    dy = G.dev(guard)
    assert call(ctypes.c_void_p(G.vp(dy).value + 2 * pad)) == 0, ghip.apus_ghip_last_error()
    got = G.host(dy, np.uint16, guard.shape)
    assert np.all(got[:pad] == 0x7E57) and np.all(got[pad + M * N:] == 0x7E57), "wrote outside y"
    return got[pad:pad + M * N].reshape(M, N)


def run_fp8(ghip, codes, scales, x, exact, pad=8):
    (N, K), M = codes.shape, x.shape[0]
    dc, ds, dx = G.dev(codes), G.dev(scales), G.dev(x)
    return guarded(ghip, lambda y: ghip.apus_ghip_fp8blk_linear_dev(
        G.vp(dc), G.vp(ds), G.vp(dx), y, M, N, K, exact, G.stream()), M, N, pad)


def fp8_inputs(M, N, K, nan_codes):
    rng = np.random.default_rng(M * 1009 + N * 13 + K)
    codes = rng.integers(0, 256 if nan_codes else 254, (N, K), dtype=np.uint8)
    if not nan_codes:
        codes[codes >= 0x7F] += 1
    scales = np.exp2(rng.uniform(-10, -4, (O.nblocks(N), O.nblocks(K)))).astype(np.float32)
    return codes, scales, O.f32_to_bf16(rng.standard_normal((M, K)).astype(np.float32))


@pytest.mark.parametrize("M,N,K", FP8)
def test_rows_fp8(ghip, M, N, K):
    """Clean codes: both decodes give the same bits; then NaN codes."""
    held_to_form(ghip, 0, M, N, K, FP8[M, N, K])
    for nan_codes in (False, True):
        codes, scales, x = fp8_inputs(M, N, K, nan_codes)
        w = O.dequant(codes, scales, threads=8)
        floor = 2.0 ** -8 * (np.abs(O.bf16_to_f32(x)) @ np.abs(O.bf16_to_f32(w)).T)
        got = run_fp8(ghip, codes, scales, x, 1)
        assert_close(got, O.gemm(w, x, threads=16), floor, "fp8 M%d N%d K%d" % (M, N, K))
        if not nan_codes:
            assert np.array_equal(got, run_fp8(ghip, codes, scales, x, 0))
            assert np.array_equal(got, run_fp8(ghip, codes, scales, x, -1, pad=1))


@pytest.mark.parametrize("M,N,K", BF16)
def test_rows_bf16(ghip, M, N, K):
    held_to_form(ghip, 1, M, N, K, BF16[M, N, K])
    check_bf16(ghip, M, N, K)


def check_bf16(ghip, M, N, K):
    rng = np.random.default_rng(M * 1013 + N * 17 + K)
    w = O.f32_to_bf16(rng.uniform(-4, 4, (N, K)).astype(np.float32))
    x = O.f32_to_bf16(rng.uniform(-4, 4, (M, K)).astype(np.float32))
    dw, dx = G.dev(w), G.dev(x)
    got = [guarded(ghip, lambda y: ghip.apus_ghip_bf16_gemm_dev(
        G.vp(dw), G.vp(dx), y, M, N, K, G.stream()), M, N, pad) for pad in (8, 1)]
    floor = 2.0 ** -8 * (np.abs(O.bf16_to_f32(x)) @ np.abs(O.bf16_to_f32(w)).T)
    assert_close(got[0], O.gemm(w, x, threads=16), floor, "bf16 M%d N%d K%d" % (M, N, K))
    assert np.array_equal(got[0], got[1])


@pytest.mark.parametrize("M,N,K", [(1, 17, 4096), (4, 288, 4160), (3, 2048, 4672), (2, 100, 4096 + 64 * 21),
                                   (4, 33, 12288), (1, 2041, 8192 + 64)])
def test_few_long_bf16_rows(ghip, M, N, K):
    """Few long weight rows (the streaming GEMV with x staged): every count of
    chunks left after its loop of three, and row remainders."""
    assert ghip.ghip_bf16_linear_route(ctypes.c_void_p(16), ctypes.c_void_p(16), ctypes.c_size_t(M), ctypes.c_size_t(N),
                                       ctypes.c_size_t(K), 256) == 1
    check_bf16(ghip, M, N, K)


def test_rows_not_finite(ghip):
    """An infinity in x reaches exactly its own row (rows past M re-read the
    last one and are not stored)."""
    codes, scales, x = fp8_inputs(5, 100, 256, False)
    codes &= 0x77                                                   # positive, finite
    codes[codes == 0] = 0x11
    x[4, 9] = 0x7F80
    y = O.bf16_to_f32(run_fp8(ghip, codes, scales, x, 0))
    assert np.all(np.isposinf(y[4])) and np.all(np.isfinite(y[:4]))


def test_rows_several_launches(ghip):
    """More rows than one launch's 65535 row tiles hold, whatever the tile:
    every row is computed once, from its own x."""
    M, N, K, period = 65535 * 64 + 5, 20, 128, 1009
    codes, scales, x = fp8_inputs(period, N, K, False)
    w = O.dequant(codes, scales, threads=8)
    floor = 2.0 ** -8 * (np.abs(O.bf16_to_f32(x)) @ np.abs(O.bf16_to_f32(w)).T)
    got = run_fp8(ghip, codes, scales, np.resize(x, (M, K)), 0)
    assert_close(got[:period], O.gemm(w, x, threads=16), floor, "first rows")
    whole = M // period * period
    assert (got[:whole].reshape(-1, period, N) == got[:period]).all()
    assert np.array_equal(got[whole:], got[:M - whole])
