"""Host-pointer calls on both sides of the size up to which x and y go through
pinned memory (256 KB each), with odd byte counts, repeated calls with other
inputs, several calls sharing the pinned memory, calls that fail with pieces
taken, and decodes of two stores from two threads: the same bits as the
device-pointer call, or as the calls alone."""
import threading

import numpy as np
import pytest

import oracle as O
import gpu_util as G
from test_gpu_moe import open_store, random_slabs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,o,k", [(1, 1, 128), (1, 7, 256), (3, 129, 128), (32, 300, 4096), (33, 300, 4096),
                                   (64, 2048, 128), (65, 2048, 128), (65, 2048, 2048), (5, 33, 77)])
def test_matches_device_call(ghip, m, o, k):
    rng = np.random.default_rng(m * 7919 + o)
    for _ in range(3):
        codes = rng.integers(0, 254, (o, k), dtype=np.uint8)
        codes[codes >= 0x7F] += 1
        scales = np.exp2(rng.uniform(-13, -7, ((o + 127) // 128, (k + 127) // 128))).astype(np.float32)
        x = O.f32_to_bf16(rng.standard_normal((m, k)).astype(np.float32))
        y = np.empty(m * o + 8, np.uint16)
        y[m * o:] = 0xABCD
        assert ghip.apus_ghip_fp8blk_linear(O.ptr(codes), O.ptr(scales), O.ptr(x), O.ptr(y), m, o, k) == 0
        dc, ds, dx, dy = G.dev(codes), G.dev(scales), G.dev(x), G.empty(m * o * 2)
        assert ghip.apus_ghip_fp8blk_linear_dev(G.vp(dc), G.vp(ds), G.vp(dx), G.vp(dy), m, o, k, 0,
                                                G.stream()) == 0
        assert np.array_equal(y[:m * o].reshape(m, o), G.host(dy, np.uint16, (m, o)))
        assert (y[m * o:] == 0xABCD).all()


def test_two_threads_two_stores(ghip):
    """Decodes of two stores at once: the pinned memory serves one of the calls
    at a time, and each gets the output of its own inputs."""
    dim, inter, E, k, n = 1024, 512, 6, 3, 300
    rng = np.random.default_rng(31)
    stores = [open_store(ghip, E, dim, inter) for _ in range(2)]
    try:
        jobs = []
        for s in stores:
            for e, sl in enumerate(random_slabs(E, dim, inter, rng)):
                assert ghip.apus_ghip_store_put(s, e, O.ptr(sl), sl.nbytes) == 0
            x = O.f32_to_bf16(rng.standard_normal((8, dim)).astype(np.float32))
            idx = np.stack([rng.permutation(E)[:k] for _ in range(8)]).astype(np.int32)
            w = rng.uniform(0.1, 0.5, (8, k)).astype(np.float32)
            jobs.append((s, x, idx, w, np.empty((8, dim), np.uint16)))

        def decode(s, x, idx, w, out):
            assert ghip.apus_ghip_moe_decode(s, O.ptr(x), O.ptr(idx), O.ptr(w), k, O.ptr(out)) == 0

        for s, x, idx, w, alone in jobs:
            for t in range(8):
                decode(s, x[t].copy(), idx[t].copy(), w[t].copy(), alone[t])
        wrong = [0, 0]

        def work(j):
            s, x, idx, w, alone = jobs[j]
            out = np.empty(dim, np.uint16)
            for i in range(n):
                t = i % 8
                decode(s, x[t].copy(), idx[t].copy(), w[t].copy(), out)
                wrong[j] += not np.array_equal(out, alone[t])
            wrong[j] += 0 if i == n - 1 else 1

        th = [threading.Thread(target=work, args=(j,)) for j in range(2)]
        for t in th:
            t.start()
        for t in th:
            t.join()
        assert wrong == [0, 0]
    finally:
        for s in stores:
            ghip.apus_ghip_store_close(s)


def test_failed_call_gives_the_pinned_memory_back(ghip):
    """A call that fails after its copies in (more than 1024 experts: refused
    at the launch) leaves none of its pieces to the next call, on this thread
    or another."""
    dim, inter, E = 256, 128, 1025
    rng = np.random.default_rng(32)
    s = open_store(ghip, E, dim, inter)
    x = O.f32_to_bf16(rng.standard_normal((2, dim)).astype(np.float32))
    idx, w, out = np.zeros((2, 1), np.int32), np.ones((2, 1), np.float32), np.empty((2, dim), np.uint16)
    try:
        fail = []
        th = threading.Thread(target=lambda: fail.append(
            ghip.apus_ghip_moe_prefill(s, O.ptr(x), 2, O.ptr(idx), O.ptr(w), 1, O.ptr(out))))
        th.start()
        th.join()
        assert fail == [1]
    finally:
        ghip.apus_ghip_store_close(s)
    test_matches_device_call(ghip, 3, 129, 128)
