"""The FP8-block GEMM on MFMA (k_fp8_gemm, csrc/k_moe_prefill.hip) behind the
fp8blk_linear entry, against the oracle to the contract tolerance
(tests/tolerance.py): each tile height with and without a K split, the bodies
of 1 to 8 row blocks, each with clean codes by both decodes (the same bits) and
with NaN codes by the exact one."""
import ctypes

import numpy as np
import pytest

import oracle as O
from test_gpu_rows import fp8_inputs, run_fp8
from tolerance import assert_close

pytestmark = pytest.mark.gpu

# (M, N, K): tile height and K splits on 256 CUs, to which each case is held
SHAPES = {(257, 256, 128): (32, 1), (257, 256, 512): (32, 2),
          (197, 12544, 128): (64, 1), (481, 512, 3072): (64, 12),           # 1 and 2 row blocks left
          (386, 12288, 128): (128, 1), (500, 12288, 128): (128, 1),         # 1 and 4
          (67, 12288, 1152): (128, 4),                                      # 3, the fourth empty
          (801, 12288, 128): (256, 1), (129, 9984, 2176): (256, 5)}         # 8 and 2; 5 of 8
GEMM = 3                                                            # the route's number (ghip_internal.h)


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_fp8_gemm_bodies(ghip, M, N, K):
    p, z = ctypes.c_void_p(1 << 20), [ctypes.c_size_t(v) for v in (M, N, K)]
    form = ghip.ghip_fp8_gemm_form(*z, 256)
    assert ghip.ghip_fp8_linear_route(p, p, p, *z, 256) == GEMM and (form >> 16, form & 0xffff) == SHAPES[M, N, K]
    for nan_codes in (False, True):
        codes, scales, x = fp8_inputs(M, N, K, nan_codes)
        w = O.dequant(codes, scales, threads=16)
        floor = 2.0 ** -8 * (np.abs(O.bf16_to_f32(x)) @ np.abs(O.bf16_to_f32(w)).T)
        got = run_fp8(ghip, codes, scales, x, 1)
        assert_close(got, O.gemm(w, x, threads=16), floor, "fp8 M%d N%d K%d" % (M, N, K))
        if not nan_codes:
            assert np.array_equal(got, run_fp8(ghip, codes, scales, x, 0))
            assert np.array_equal(got, run_fp8(ghip, codes, scales, x, -1))
