"""The BF16-weight GEMM on MFMA (csrc/k_gemm_bf16.hip) behind the bf16_gemm
entry, against the oracle's sequential-k GEMM to the contract tolerance
(tests/tolerance.py): every tile shape the launcher picks, ring lengths below,
at and above the pipeline's depth (K = 64 is one stage), row and column
remainders, and result rows that do not allow vector stores."""
import ctypes

import numpy as np
import pytest

import oracle as O
import gpu_util as G
from tolerance import assert_close

pytestmark = pytest.mark.gpu

# (M, N, K): the tile the library picks on 256 CUs, to which each case is held
SHAPES = {(65, 8000, 64): (64, 64), (250, 2050, 128): (64, 64), (130, 4100, 1088): (64, 64),
          (64, 20000, 192): (64, 128), (320, 4000, 448): (64, 128),
          (600, 4096, 320): (192, 64),
          (1023, 4095, 128): (128, 128), (1024, 4096, 704): (128, 128),
          (1100, 4104, 256): (192, 128),
          (2047, 4096, 320): (256, 128),
          (2048, 8185, 192): (256, 256)}
GEMM = 3                                                            # the route's number (ghip_internal.h)


def on_gemm(ghip, M, N, K):
    p, z = ctypes.c_void_p(1 << 20), [ctypes.c_size_t(v) for v in (M, N, K)]
    assert ghip.ghip_bf16_linear_route(p, p, *z, 256) == GEMM
    form = ghip.ghip_bf16_gemm_form(z[0], z[1], 256)
    return form >> 16, form & 0xffff


def run(ghip, w, x, pad):
    """y through the device entry, inside a guarded buffer `pad` elements in."""
    (N, K), M = w.shape, x.shape[0]
    guard = np.full(M * N + 64, 0x7E57, np.uint16)
    dw, dx, dy = G.dev(w), G.dev(x), G.dev(guard)
    yp = ctypes.c_void_p(G.vp(dy).value + 2 * pad)
    assert ghip.apus_ghip_bf16_gemm_dev(G.vp(dw), G.vp(dx), yp, M, N, K, G.stream()) == 0, \
        ghip.apus_ghip_last_error()
    got = G.host(dy, np.uint16, guard.shape)
    assert np.all(got[:pad] == 0x7E57) and np.all(got[pad + M * N:] == 0x7E57), "wrote outside y"
    return got[pad:pad + M * N].reshape(M, N)


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_bf16_gemm_tiles(ghip, M, N, K):
    assert on_gemm(ghip, M, N, K) == SHAPES[M, N, K]
    rng = np.random.default_rng(M * 31 + N * 7 + K)
    w = O.f32_to_bf16(rng.uniform(-4, 4, (N, K)).astype(np.float32))
    x = O.f32_to_bf16(rng.uniform(-4, 4, (M, K)).astype(np.float32))
    got = run(ghip, w, x, 8)
    floor = 2.0 ** -8 * (np.abs(O.bf16_to_f32(x)) @ np.abs(O.bf16_to_f32(w)).T)
    assert_close(got, O.gemm(w, x, threads=16), floor, "bf16 M%d N%d K%d" % (M, N, K))
    assert np.array_equal(got, run(ghip, w, x, 8))                  # deterministic


def test_bf16_gemm_unaligned_y(ghip):
    """y two bytes off a 16-byte boundary: the same values by 2-byte stores."""
    rng = np.random.default_rng(11)
    on_gemm(ghip, 250, 2056, 256)
    w = O.f32_to_bf16(rng.uniform(-4, 4, (2056, 256)).astype(np.float32))
    x = O.f32_to_bf16(rng.uniform(-4, 4, (250, 256)).astype(np.float32))
    assert np.array_equal(run(ghip, w, x, 1), run(ghip, w, x, 8))


def test_bf16_gemm_not_finite(ghip):
    """An infinity and a NaN reach exactly their own row or column (rows past
    M and N re-read the last one and are not stored)."""
    rng = np.random.default_rng(12)
    M, N, K = 250, 2050, 128
    on_gemm(ghip, M, N, K)
    w = O.f32_to_bf16(rng.uniform(1, 4, (N, K)).astype(np.float32))
    x = O.f32_to_bf16(rng.uniform(1, 4, (M, K)).astype(np.float32))
    x[M - 1, 5], w[N - 1, 7] = 0x7F80, 0x7FC0                       # +inf, NaN
    y = O.bf16_to_f32(run(ghip, w, x, 8))
    assert np.all(np.isnan(y[:, N - 1])) and np.all(np.isposinf(y[M - 1, :N - 1]))
    assert np.all(np.isfinite(y[:M - 1, :N - 1]))
