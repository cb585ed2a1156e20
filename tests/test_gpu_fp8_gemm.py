"""The FP8-block GEMM on MFMA (k_fp8_gemm, csrc/k_moe_prefill.hip) behind the
fp8blk_linear entry, against the oracle to the contract tolerance
(tests/tolerance.py): each tile height with and without a K split, the bodies
of 1 to 8 row blocks, each with clean codes by both decodes (the same bits) and
with NaN codes by the exact one."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

import gpu_util as G
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


def split_bytes(ghip, M, N, K):
    p, z = ctypes.c_void_p(1 << 20), [ctypes.c_size_t(v) for v in (M, N, K)]
    assert ghip.ghip_fp8_linear_route(p, p, p, *z, 256) == GEMM
    splits = ghip.ghip_fp8_gemm_form(*z, 256) & 0xffff
    return splits * M * N * 4 if splits > 1 else 0


def child_captures_splits():
    """The buffer of the K splits and graphs, from the process's first call:
    a capture that cannot allocate it takes the form without splits; one that
    holds it replays the same bits after eager calls have grown the buffer
    twice, and writes into none of the memory allocated since."""
    from conftest import load_pkg
    ghip = load_pkg().load()
    err = ctypes.create_string_buffer(256)
    assert ghip.apus_ghip_enable(err, 256) == 0, err.value
    M, N, K = 168, 1536, 8192
    need = split_bytes(ghip, M, N, K)
    assert need
    codes, scales, x = fp8_inputs(M, N, K, False)
    w = O.dequant(codes, scales, threads=16)
    floor = 2.0 ** -8 * (np.abs(O.bf16_to_f32(x)) @ np.abs(O.bf16_to_f32(w)).T)
    want = O.gemm(w, x, threads=16)
    dc, ds, dx, dy = G.dev(codes), G.dev(scales), G.dev(x), G.empty(M * N * 2)
    rt = G.rt()
    st = rt.Stream()

    def call():
        return ghip.apus_ghip_fp8blk_linear_dev(G.vp(dc), G.vp(ds), G.vp(dx), G.vp(dy), M, N, K, 0,
                                                st.vp)

    def out():
        st.synchronize()
        y = G.host(dy, np.uint16, (M, N))
        dy.zero()
        rt.synchronize()
        return y

    def captured():
        g = rt.Graph(st)
        g.begin()
        try:
            rc = call()
        finally:
            g.end()
        assert rc == 0, ghip.apus_ghip_last_error()
        return g

    first = captured()
    first.launch()
    bare = out()
    assert_close(bare, want, floor, "captured before any split")
    assert call() == 0, ghip.apus_ghip_last_error()
    eager = out()
    assert_close(eager, want, floor, "eager")
    assert not np.array_equal(eager, bare)              # the other form's order of sums
    second = captured()
    kept = []
    for rows in (168, 400, 1600):
        if rows > M:
            more = split_bytes(ghip, rows, N, K)
            assert more > need
            need = more
            c2, s2, x2 = codes, scales, fp8_inputs(rows, N, K, False)[2]
            y2 = run_fp8(ghip, c2, s2, x2, 0)
            assert_close(y2[:32], O.gemm(w, x2[:32], threads=16),
                         2.0 ** -8 * (np.abs(O.bf16_to_f32(x2[:32])) @ np.abs(O.bf16_to_f32(w)).T),
                         "eager %d rows" % rows)
            kept += [G.dev(np.full(12 << 20, 0x5A, np.uint8)) for _ in range(4)]
        for g, ref in ((second, eager), (first, bare), (second, eager)):
            g.launch()
            assert np.array_equal(out(), ref), rows
        for b in kept:
            assert (G.host(b, np.uint8, (12 << 20,)) == 0x5A).all()
    for g in (first, second):
        g.close()
    print("captures of K splits ok", flush=True)


def test_fp8_gemm_splits_under_capture():
    """In a process of its own: the library's first FP8 product is captured."""
    here = os.path.dirname(os.path.abspath(__file__))
    code = ("import sys; sys.path[:0] = [%r, %r]; import test_gpu_fp8_gemm as t; "
            "t.child_captures_splits()" % (here, os.path.join(os.path.dirname(here), "oracle")))
    p = subprocess.run([sys.executable, "-c", code], stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=100)
    assert p.returncode == 0 and "captures of K splits ok" in p.stdout, p.stdout
