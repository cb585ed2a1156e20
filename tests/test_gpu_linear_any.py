"""The shape-general linear (K no multiple of 128 or 64), which takes 1, 2, 4
or 8 rows of x a wave: row remainders at each, K under one wave's step, one to
four steps of 64 left after those of 256, full and partial, and scale blocks
crossed inside one; against the oracle to
the contract tolerance, and the same bits for a row whatever rows are beside
it."""
import numpy as np
import pytest

import oracle as O
import gpu_util as G
from test_gpu_rows import fp8_inputs, guarded, run_fp8
from tolerance import assert_close

pytestmark = pytest.mark.gpu

SIZES = [(1, 5, 1), (1, 4097, 63), (2, 4100, 65), (3, 2050, 255), (4, 5000, 257), (7, 4099, 100),
         (8, 4096, 191), (9, 2100, 449), (17, 1500, 330), (64, 700, 1025), (33, 64, 500),
         (3, 2000, 257), (5, 300, 447), (6, 300, 576 + 32), (2, 500, 1216 + 32)]


@pytest.mark.parametrize("M,N,K", SIZES)
def test_any_fp8(ghip, M, N, K):
    codes, scales, x = fp8_inputs(M, N, K, True)
    w = O.dequant(codes, scales, threads=8)
    floor = 2.0 ** -8 * (np.abs(O.bf16_to_f32(x)) @ np.abs(O.bf16_to_f32(w)).T)
    got = run_fp8(ghip, codes, scales, x, 0)
    assert_close(got, O.gemm(w, x, threads=16), floor, "fp8 M%d N%d K%d" % (M, N, K))
    assert np.array_equal(got[-1:], run_fp8(ghip, codes, scales, x[-1:].copy(), 0))


@pytest.mark.parametrize("M,N,K", SIZES)
def test_any_bf16(ghip, M, N, K):
    rng = np.random.default_rng(M * 1013 + N * 17 + K)
    w = O.f32_to_bf16(rng.uniform(-4, 4, (N, K)).astype(np.float32))
    x = O.f32_to_bf16(rng.uniform(-4, 4, (M, K)).astype(np.float32))

    def run(x):
        dw, dx = G.dev(w), G.dev(x)
        return guarded(ghip, lambda y: ghip.apus_ghip_bf16_gemm_dev(
            G.vp(dw), G.vp(dx), y, len(x), N, K, G.stream()), len(x), N, 1)

    got = run(x)
    floor = 2.0 ** -8 * (np.abs(O.bf16_to_f32(x)) @ np.abs(O.bf16_to_f32(w)).T)
    assert_close(got, O.gemm(w, x, threads=16), floor, "bf16 M%d N%d K%d" % (M, N, K))
    assert np.array_equal(got[-1:], run(x[-1:].copy()))


def test_any_several_launches(ghip):
    """More waves than one launch holds (2^32 threads): every output is
    written. K = 1, so an output is one product."""
    M, N = 65541, 8200
    assert -(-M // 8) * N * 64 > 1 << 32
    rng = np.random.default_rng(4)
    w = O.f32_to_bf16(rng.uniform(-4, 4, (N, 1)).astype(np.float32))
    x = O.f32_to_bf16(rng.uniform(-4, 4, (M, 1)).astype(np.float32))
    dw, dx, dy = G.dev(w), G.dev(x), G.empty(2 * M * N)
    assert ghip.apus_ghip_bf16_gemm_dev(G.vp(dw), G.vp(dx), G.vp(dy), M, N, 1, G.stream()) == 0
    got = G.host(dy, np.uint16, (M, N))
    for m in range(0, M, 4096):
        want = O.f32_to_bf16(O.bf16_to_f32(x[m:m + 4096]) * O.bf16_to_f32(w).T + np.float32(0))
        assert np.array_equal(got[m:m + 4096], want), m
